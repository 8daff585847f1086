// fp32 projections straight from memory into fp32 MFMA operands.
//
//   out[M x N] = A[M x K] . W[K x N]              one or two segments side by side
//   out[M x N] = SiLU(A0 . W0) * (A1 . W1)        DUAL: the two branches of a tile
//
// The fp32 MFMA (16x16x4, 64 FLOP per cycle and SIMD) is slow enough that its
// operands need no LDS: a wave's 16 MT x 64 tile takes 4 KB of weights and MT
// KB of activations per 16 k against 512 MT matrix cycles, 16 to 24 bytes per
// cycle and CU, which the caches deliver.
//  * One 16-byte load per lane is four operands as it lies: natural layout,
//    lane (lr, lg) reads columns 4 lr .. + 3 of row k0 + 4 lg + i, operand
//    (i, c) holding column 4 lr + c; Linear layout, k0 + 4 lg .. + 3 of row
//    4 lr + c; activations k0 + 4 lg .. + 3 of token row lr.
//  * A block's 8 waves split K (DUAL: four waves a branch) and meet in LDS;
//    further K splits over blocks meet through slices summed in split order
//    by the last block to arrive (stream.hpp), so small layers fill the
//    chip: the (128, 1024, 3584, 256) layer's stages have 4 to 28 tiles of
//    128 x 128.
//  * Transposed operands ((K, M) activations, (N, M) results) are read and
//    written as they lie, 64 bytes of a row at a time.
// Measured against the LDS-tiled 128 x 128 kernel (256-thread blocks, K
// splits summed by float atomics) it replaced, rotating weights: (1024, 3584,
// 256) at 1 / 128 / 1024 / 4096 tokens 163 / 186 / 208 / 456 -> 23 / 30 / 89 /
// 295 us, (2048, 5632, 1152) at 128 / 2048 tokens 426 / 1331 -> 122 / 898 us
// (102 TFLOP/s; a large fp32 matrix product reaches 153 here).
#pragma once

#include "stream.hpp"

namespace svdmlp {

struct StreamF32Seg {
  const float* a;  // (M, K), row pitch K, or with AT (K, M)
  const float* w;  // (K, N), or (N, K) in the Linear layout
  float* out;      // (M, N), row pitch N, or with out_t (N, M)
  int64_t ldw;
  int K, N;
  int ntiles;      // ceil(N / 64)
  int ks;          // K per split, a multiple of 16
};

struct StreamF32Params {
  StreamF32Seg seg[2];
  int M, splits, tiles, mtiles;  // tiles: column tiles over the segments (DUAL: of one)
  float* slices;                 // (tile, split, branch) slices of 16 MT x 64
  uint32_t slice_bytes;
  uint64_t* sync;
  const float* resid;            // (M, N) added to out, or null
  int out_t;                     // out is (N, M)
};

constexpr int kSfTileN = 64;

template <int MT>
struct SfStep {
  f32x4 w[4], a[MT];
};

template <int MT, bool LIN, bool AT>
__device__ __forceinline__ void sf_load(const StreamF32Seg& s, int M, int m0, int n0, int k0, bool live, int lr, int lg,
                                        SfStep<MT>& r) {
  const int records = live ? 0x7ffffff0 : 0;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(s.a) + (AT ? (int64_t)k0 * M + m0 : (int64_t)m0 * s.K + k0), 0, records, 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(s.w) + (LIN ? (int64_t)n0 * s.ldw + k0 : (int64_t)k0 * s.ldw + n0), 0, records, 0x00020000);
  const uint32_t ld = live ? (uint32_t)s.ldw * 4u : 0u;
  // K and N are multiples of 4: a lane's piece is inside or outside as a whole
  const uint32_t k_past = k0 + 4 * lg < s.K ? 0u : kOOB;
  const uint32_t v = ((LIN ? (uint32_t)(4 * lr) * ld + 16u * lg : (uint32_t)(4 * lg) * ld + 16u * lr)) | k_past |
                     (n0 + 4 * lr < s.N ? 0u : kOOB);
#pragma unroll
  for (int j = 0; j < 4; ++j) r.w[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, v, j * ld, 0));
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = 16 * mt + lr;
    if constexpr (AT) {
      const uint32_t off = ((uint32_t)(4 * lg) * (uint32_t)M + (uint32_t)m) * 4u | k_past | (m0 + m < M ? 0u : kOOB);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        r.a[mt][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ra, off, live ? (uint32_t)(i * M) * 4u : 0u, 0));
      continue;
    }
    const uint32_t row = m0 + m < M ? (uint32_t)m * (uint32_t)s.K * 4u : kOOB;
    r.a[mt] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ra, (row + 16u * lg) | k_past, 0, 0));
  }
}

// acc[mt][c]: token rows 16 mt .., columns 4 lr + c.
template <int MT, bool LIN>
__device__ __forceinline__ void sf_mul(const SfStep<MT>& r, f32x4 (&acc)[MT][4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        acc[mt][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(r.a[mt][i], LIN ? r.w[c][i] : r.w[i][c], acc[mt][c], 0, 0, 0);
}

template <int MT, bool LIN, bool DUAL, bool AT>
__global__ __launch_bounds__(kStThreads, 2) void stream_f32_kernel(StreamF32Params p) {
  constexpr int NWB = DUAL ? 4 : 8;  // waves per branch
  constexpr int BR = DUAL ? 2 : 1;
  constexpr int PITCH = kSfTileN;
  __shared__ __attribute__((aligned(16))) float red[8][16 * PITCH];
  __shared__ int last;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane & 15, lg = lane >> 4;
  int splits = p.splits, nt0 = p.seg[0].ntiles;
  asm volatile("" : "+s"(splits), "+s"(nt0));  // loaded with the other arguments, not on their own later

  // blocks in (split, column tile, row tile) order: the row tiles of a column
  // tile read the same weights
  const int all = p.tiles * p.mtiles;
  const int split = blockIdx.x / all, t0 = blockIdx.x % all;
  const int tile = t0 / p.mtiles, m0 = t0 % p.mtiles * (16 * MT);
  const bool second = !DUAL && tile >= nt0;
  const StreamF32Seg& so = p.seg[second ? 1 : 0];
  const StreamF32Seg& s = p.seg[DUAL ? wave >> 2 : (second ? 1 : 0)];
  const int n0 = (second ? tile - nt0 : tile) * kSfTileN;
  const int kb = split * s.ks, ke = min(s.K, kb + s.ks);
  const int wb = DUAL ? wave & 3 : wave;

  // after a timeout on the workspace (its tile counters are in an unknown state)
  // the first split's block takes its tile's whole K (stream.hpp)
  const uint32_t flag = __hip_atomic_load(reinterpret_cast<uint32_t*>(&p.sync[kDlFlag]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  f32x4 acc[MT][4];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[mt][c] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto run = [&](int kb, int ke) {
    const int nst = (ke - kb + 15) / 16;
    const int steps = nst > wb ? (nst - wb + NWB - 1) / NWB : 0;
    SfStep<MT> r0, r1;
    auto load = [&](int i, SfStep<MT>& r) {
      sf_load<MT, LIN, AT>(s, p.M, m0, n0, kb + 16 * (i * NWB + wb), i < steps, lr, lg, r);
    };
    load(0, r0);
    for (int i = 0; i < steps; i += 2) {
      load(i + 1, r1);
      __builtin_amdgcn_sched_barrier(0);
      sf_mul<MT, LIN>(r0, acc);
      __builtin_amdgcn_sched_barrier(0);
      load(i + 2, r0);
      __builtin_amdgcn_sched_barrier(0);
      sf_mul<MT, LIN>(r1, acc);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  run(kb, ke);
  if (splits > 1 && __builtin_amdgcn_readfirstlane(flag)) {
    if (split) return;
    run(ke, s.K);
    splits = 1;
  }

  auto finish = [&](int m, int n, f32x4 v0, f32x4 v1) {
    if constexpr (DUAL)
      v0 = f32x4{silu_f32(v0.x) * v1.x, silu_f32(v0.y) * v1.y, silu_f32(v0.z) * v1.z, silu_f32(v0.w) * v1.w};
    const int64_t off = (int64_t)m * so.N + n0 + n;
    if (p.out_t) {
#pragma unroll
      for (int i = 0; i < 4; ++i) so.out[(int64_t)(n0 + n + i) * p.M + m] = v0[i];
      return;
    }
    if (p.resid) v0 = *reinterpret_cast<const f32x4*>(p.resid + off) + v0;
    *reinterpret_cast<f32x4*>(so.out + off) = v0;
  };

  // ---- the 8 waves' sums, 16 token rows at a time: thread (half tid / 256,
  // row (tid / 16) % 16, columns 4 (tid % 16)..) adds one half of the waves
  // (DUAL: one branch), and the second half's threads hand theirs over ----
  const int half = tid >> 8, qm = (tid >> 4) & 15, qn = 4 * (tid & 15);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(p.slices, 0, (int)p.slice_bytes, 0x00020000);
  const uint32_t unit = (uint32_t)(t0 * p.splits + split) * BR;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    if (m0 + 16 * mt < p.M) {  // uniform
      __syncthreads();
#pragma unroll
      for (int t = 0; t < 4; ++t)
        *reinterpret_cast<f32x4*>(&red[wave][(4 * lg + t) * PITCH + 4 * lr]) =
            f32x4{acc[mt][0][t], acc[mt][1][t], acc[mt][2][t], acc[mt][3][t]};
      __syncthreads();
      f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < 4; ++w) v += *reinterpret_cast<const f32x4*>(&red[4 * half + w][qm * PITCH + qn]);
      const int m = m0 + 16 * mt + qm;
      const bool in = m < p.M && n0 + qn < so.N;
      if (DUAL && splits > 1) {
        if (in)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rs,
                                                 (((unit + half) * (16 * MT) + (16 * mt + qm)) * kSfTileN + qn) * 4u, 0, kDlSc1);
      } else {
        __syncthreads();  // every wave's part is read
        f32x4* const hand = reinterpret_cast<f32x4*>(&red[0][0]);
        if (half) hand[tid & 255] = v;
        __syncthreads();
        if (!half && in) {
          const f32x4 o = hand[tid];
          if (splits > 1)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v + o), rs,
                                                   ((unit * (16 * MT) + (16 * mt + qm)) * kSfTileN + qn) * 4u, 0, kDlSc1);
          else if (DUAL)
            finish(m, qn, v, o);
          else
            finish(m, qn, v + o, o);
        }
      }
    }
  }
  if (splits == 1) return;

  // ---- K splits: the last block of the tile to arrive sums the slices in
  // split order ----
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0)
    last = __builtin_amdgcn_atomic_inc32(dl_tile_counter(p.sync, t0), (uint32_t)splits - 1u, __ATOMIC_RELAXED, "agent") ==
           (uint32_t)splits - 1u;
  __syncthreads();
  if (!last) return;
  const uint32_t unit0 = (uint32_t)(t0 * p.splits) * BR;
  constexpr int SB = DUAL ? 4 : 8;  // splits in flight
  for (int q = tid; q < 16 * MT * 16; q += kStThreads) {
    const int m = m0 + (q >> 4), n = 4 * (q & 15);
    if (m >= p.M || n0 + n >= so.N) continue;
    f32x4 v[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    for (int s0 = 0; s0 < splits; s0 += SB) {
      f32x4 x[SB][BR];
#pragma unroll
      for (int k = 0; k < SB; ++k)
#pragma unroll
        for (int b = 0; b < BR; ++b)
          x[k][b] = __builtin_bit_cast(
              f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                         rs, s0 + k < splits ? (unit0 + (uint32_t)((s0 + k) * BR + b)) * (16u * MT * kSfTileN * 4u) + 16u * (uint32_t)q
                                               : kStNone,
                         0, kDlSc1));
#pragma unroll
      for (int k = 0; k < SB; ++k)
#pragma unroll
        for (int b = 0; b < BR; ++b) v[b] += x[k][b];
    }
    finish(m, n, v[0], v[1]);
  }
}

}  // namespace svdmlp
