// Streaming stages (stream.hpp) of Linear-layout bf16 weights at one or two
// tokens: a row of W is a column of the result, so a wave takes two columns
// over their whole K with coalesced 16-byte loads (64 lanes, 512 k a step) and
// fp32 multiply-adds, and sums its lanes' parts.  No K split, no slices, no
// LDS and no counter.
//
// Bound by the weight stream, and in small layers by the latency of a launch.
// The MFMA stages spend that on sums in LDS, slices, arrivals and the last
// unit's sums, and their tiles of 128 columns are too coarse for the CUs in a
// small layer.  us per layer at 1 / 2 tokens, MFMA stages -> these: (4096,
// 14336, 2816) 77.5 / 77.3 -> 65.9 / 73.6, (3072, 8192, 1792) 46.4 / 46.5 ->
// 32.2 / 37.2, (2048, 5632, 1152) 37.9 / 37.5 -> 22.3 / 26.7, (1024, 3584,
// 256) 30.0 / 29.9 -> 20.2 / 20.6.  The multiply-adds grow with the tokens
// where the MFMA stages' time does not (8B 7.7 us a token, 78.3 us there at
// three): the line is at two.
#include "stream.hpp"

#include "dispatch.hpp"

namespace svdmlp {

namespace {

constexpr int kGlCols = 2;  // columns a wave

template <int T, bool DUAL>
__global__ __launch_bounds__(64) void gemv_linear_kernel(StreamParams p) {
  constexpr int BR = DUAL ? 2 : 1;
  constexpr int U = DUAL ? 2 : 4;  // 512-k steps in a batch; two batches' registers alternate
  const int lane = threadIdx.x;
  const int g0 = p.seg[0].N / kGlCols;
  const bool second = !DUAL && (int)blockIdx.x >= g0;
  const StreamSeg& so = p.seg[second ? 1 : 0];
  const int n0 = kGlCols * ((int)blockIdx.x - (second ? g0 : 0));
  const int K = so.K;  // (both branches')

  struct Batch {
    u32x4 w[U][BR][kGlCols], a[U][BR][T];
  };
  __amdgpu_buffer_rsrc_t rw[BR], ra[BR];
#pragma unroll
  for (int b = 0; b < BR; ++b) {
    const StreamSeg& s = p.seg[DUAL ? b : (second ? 1 : 0)];
    rw[b] = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(static_cast<const char*>(s.w) + (int64_t)n0 * s.ldw * 2), 0, kGlCols * K * 2, 0x00020000);
    ra[b] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(s.a), 0, T * K * 2, 0x00020000);
  }
  auto load = [&](int k0, Batch& r) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + 512 * u + 8 * lane;
      const uint32_t off = k < K ? 2u * (uint32_t)k : kOOB;  // K % 8 == 0: a piece is inside or outside as a whole
#pragma unroll
      for (int b = 0; b < BR; ++b) {
#pragma unroll
        for (int c = 0; c < kGlCols; ++c)
          r.w[u][b][c] = __builtin_amdgcn_raw_buffer_load_b128(rw[b], off, c * K * 2, 0);
#pragma unroll
        for (int t = 0; t < T; ++t) r.a[u][b][t] = __builtin_amdgcn_raw_buffer_load_b128(ra[b], off, t * K * 2, 0);
      }
    }
  };
  float acc[BR][kGlCols][T] = {};
  auto mul = [&](const Batch& r) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int b = 0; b < BR; ++b)
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float lo = __uint_as_float(r.a[u][b][t][i] << 16), hi = __uint_as_float(r.a[u][b][t][i] & 0xffff0000u);
#pragma unroll
            for (int c = 0; c < kGlCols; ++c) {
              const uint32_t w = r.w[u][b][c][i];
              acc[b][c][t] = fmaf(__uint_as_float(w << 16), lo, acc[b][c][t]);
              acc[b][c][t] = fmaf(__uint_as_float(w & 0xffff0000u), hi, acc[b][c][t]);
            }
          }
  };
  Batch r0, r1;
  load(0, r0);
  for (int k0 = 0; k0 < K; k0 += 2 * 512 * U) {
    load(k0 + 512 * U, r1);
    __builtin_amdgcn_sched_barrier(0);
    mul(r0);
    __builtin_amdgcn_sched_barrier(0);
    load(k0 + 2 * 512 * U, r0);
    __builtin_amdgcn_sched_barrier(0);
    mul(r1);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int d = 32; d; d >>= 1)
#pragma unroll
    for (int b = 0; b < BR; ++b)
#pragma unroll
      for (int c = 0; c < kGlCols; ++c)
#pragma unroll
        for (int t = 0; t < T; ++t) acc[b][c][t] += __shfl_xor(acc[b][c][t], d);
  if (lane >= T) return;
  float v[kGlCols];
#pragma unroll
  for (int c = 0; c < kGlCols; ++c) {
    v[c] = T == 2 && lane ? acc[0][c][T - 1] : acc[0][c][0];
    if constexpr (DUAL) v[c] = silu_f32(v[c]) * (T == 2 && lane ? acc[1][c][T - 1] : acc[1][c][0]);
  }
  uint32_t o = pack_bf16x2(v[0], v[1]);
  if (p.resid) o = add_bf16x2(*reinterpret_cast<const uint32_t*>(p.resid + (int64_t)lane * so.ldo + n0), o);
  *reinterpret_cast<uint32_t*>(so.out + (int64_t)lane * so.ldo + n0) = o;
}

}  // namespace

hipError_t launch_gemv_linear(const StreamParams& p, int nseg, bool dual, hipStream_t st, const char** why) {
  if (p.T < 1 || p.T > kGlMaxT || p.out_t || nseg < 1 || nseg > 2 || (dual && nseg != 2) || p.seg[0].K % 8 ||
      p.seg[0].N % 8 || (nseg == 2 && (p.seg[1].K != p.seg[0].K || p.seg[1].N % 8 || (dual && p.seg[1].N != p.seg[0].N)))) {
    *why = "Linear GEMV stage: token count, layout or dimensions outside the kernel's range";
    return hipErrorInvalidValue;
  }
  const dim3 grid((p.seg[0].N + (nseg == 2 && !dual ? p.seg[1].N : 0)) / kGlCols);
  if (p.T == 1) {
    if (dual)
      hipLaunchKernelGGL((gemv_linear_kernel<1, true>), grid, dim3(64), 0, st, p);
    else
      hipLaunchKernelGGL((gemv_linear_kernel<1, false>), grid, dim3(64), 0, st, p);
  } else {
    if (dual)
      hipLaunchKernelGGL((gemv_linear_kernel<2, true>), grid, dim3(64), 0, st, p);
    else
      hipLaunchKernelGGL((gemv_linear_kernel<2, false>), grid, dim3(64), 0, st, p);
  }
  return hipGetLastError();
}

}  // namespace svdmlp
