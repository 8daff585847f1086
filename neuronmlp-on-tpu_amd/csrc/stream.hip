// Instances and launcher of the decode-shape streaming stages (stream.hpp).
#include "stream.hpp"

#include <algorithm>

#include "dispatch.hpp"

namespace svdmlp {

namespace {

template <int MT, int WK, int CG = 1>
hipError_t go(const StreamParams& p, bool dual, hipStream_t st) {
  const dim3 grid(p.tiles * p.splits, p.groups);
  if (dual)
    hipLaunchKernelGGL((stream_kernel<MT, WK, CG, true>), grid, dim3(kStThreads), 0, st, p);
  else
    hipLaunchKernelGGL((stream_kernel<MT, WK, CG, false>), grid, dim3(kStThreads), 0, st, p);
  return hipGetLastError();
}

template <int MT>
hipError_t go_w(const StreamParams& p, int wk, int cg, bool dual, hipStream_t st) {
  if (wk == SW_LINEAR) return go<MT, SW_LINEAR>(p, dual, st);
  if constexpr (MT <= 2)
    if (wk == SW_FP8 && cg == 2) return go<MT, SW_FP8, 2>(p, dual, st);
  if (wk == SW_FP8) return go<MT, SW_FP8>(p, dual, st);
  return go<MT, SW_NATURAL>(p, dual, st);
}

}  // namespace

hipError_t launch_stream(const StreamParams& p, int wk, int cg, bool dual, hipStream_t st, const char** why) {
  if (p.T < 1 || p.T > kStMaxT || p.tiles < 1 || p.splits < 1 || p.groups != (p.T + kStRows - 1) / kStRows ||
      (p.splits > 1 && p.groups * p.tiles > kDlMaxTiles) || (cg != 1 && (wk != SW_FP8 || cg != 2 || p.T > 32))) {
    *why = "streaming stage: token count, tiles, splits or column groups outside the kernel's range";
    return hipErrorInvalidValue;
  }
  if ((p.splits > 1 || p.out_t) && (int64_t)p.groups * p.tiles * p.splits * (dual ? 2 : 1) * cg * std::min(p.T, kStRows) * kStTileN * 4 > (int64_t)p.slice_bytes) {
    *why = "streaming stage: the K splits' slices exceed the workspace's area";
    return hipErrorInvalidValue;
  }
  if (p.T <= 16) return go_w<1>(p, wk, cg, dual, st);
  if (p.T <= 32) return go_w<2>(p, wk, cg, dual, st);
  return go_w<4>(p, wk, cg, dual, st);
}

}  // namespace svdmlp
