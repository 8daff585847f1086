// Instances and launcher of the fp32 streaming stages (stream_f32.hpp).
#include "stream_f32.hpp"

#include "dispatch.hpp"

namespace svdmlp {

namespace {

template <int MT>
hipError_t go(const StreamF32Params& p, bool lin, bool dual, bool at, hipStream_t st) {
  const dim3 grid(p.tiles * p.mtiles * p.splits);
  return expand_bool(lin, [&](auto l) {
    constexpr bool L = decltype(l)::value;
    if (dual)
      hipLaunchKernelGGL((stream_f32_kernel<MT, L, true, false>), grid, dim3(kStThreads), 0, st, p);
    else if (at)
      hipLaunchKernelGGL((stream_f32_kernel<MT, L, false, true>), grid, dim3(kStThreads), 0, st, p);
    else
      hipLaunchKernelGGL((stream_f32_kernel<MT, L, false, false>), grid, dim3(kStThreads), 0, st, p);
    return hipGetLastError();
  });
}

}  // namespace

hipError_t launch_stream_f32(const StreamF32Params& p, int mt, bool lin, bool dual, bool at, hipStream_t st, const char** why) {
  if (p.M < 1 || (dual && at) || p.tiles < 1 || p.splits < 1 || p.M >= 1 << 25 || p.mtiles != (p.M + 16 * mt - 1) / (16 * mt) ||
      (int64_t)p.tiles * p.mtiles * p.splits >= (int64_t)1 << 31 ||
      (p.splits > 1 && ((int64_t)p.tiles * p.mtiles > kDlMaxTiles ||
                        (int64_t)p.tiles * p.mtiles * p.splits * (dual ? 2 : 1) * (16 * mt) * kSfTileN * 4 > (int64_t)p.slice_bytes))) {
    *why = "fp32 streaming stage: rows, tiles or splits outside the kernel's range";
    return hipErrorInvalidValue;
  }
  if (mt == 1) return go<1>(p, lin, dual, at, st);
  if (mt == 2) return go<2>(p, lin, dual, at, st);
  if (mt == 4) return go<4>(p, lin, dual, at, st);
  *why = "fp32 streaming stage: 1, 2 or 4 token tiles a block";
  return hipErrorInvalidValue;
}

}  // namespace svdmlp
