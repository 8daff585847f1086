// Decode-shape (T <= 128 tokens) projections as one launch per stage: weight
// streaming at HBM rate for the operands the persistent decode layer does not
// take (Linear-layout and fp8 factors, dimensions off its tiles) and for the
// gate/up and x.u.v entry points, which run only half of the layer.
//
//   out[T x N] = bf16(A[T x K] . W[K x N] * scale)         one or two segments side by side
//   out[T x N] = bf16(SiLU(A0 . W0) * (A1 . W1))           DUAL: the two branches of a column tile
//
// A launch is bound by the weight stream (the factors dominate every byte at
// these token counts), so the kernel keeps HBM busy and nothing else on the
// way:
//  * Weights and activations go straight from memory into MFMA operand
//    registers; no LDS and no barrier in the k loop.  A unit is a tile of 128
//    columns over one K split; its 8 waves take its 64-k blocks in turn, each
//    wave over all 128 columns, so activations are read once per block (split
//    over columns instead, every wave would read all of them).  Two steps'
//    registers alternate: while one is multiplied the other is in flight, 8
//    to 16 KB per wave, 128 KB per CU.
//  * Natural layout (K x N): lane (lr = lane % 16, lg = lane / 16) reads
//    columns 8 lr .. 8 lr + 7 of rows 8 lg .. 8 lg + 7 of a 32-k step, 16
//    lanes covering 256 (bf16) or 128 (fp8) contiguous bytes of a row; the
//    8 x 8 block is transposed with byte permutes into eight MFMA operands,
//    operand j holding column 8 lr + j.  fp8 is widened to bf16 by the
//    hardware conversion, exactly.  Linear layout (N x K): operand j is 16
//    bytes of row 8 lr + j as stored.
//  * The waves' sums meet in LDS once per unit, 16 token rows at a time.
//  * K splits: every unit stores its fp32 sums as a slice and counts its
//    arrival on the tile's counter; the last unit to arrive sums the slices
//    in split order and writes the tile.  No unit waits for another, so a
//    launch needs no resident grid (unlike the persistent decode layer) and
//    may share the device with other work, and replays are bitwise
//    identical.  No zero fill and no conversion pass: the stage before writes
//    the bf16 this stage reads.
// Measured (rotating weights, against the kernels before this one: register
// loads of a whole slice and then its MFMAs, software fp8 widening, LDS and
// global float atomics, zero-fill and conversion passes): 70B fp8 layer at 4
// tokens 800 -> 130 us (623 MB; its XU.V stage streams 323 MB in 61.0 us on
// average, 5.3 TB/s, reading 1.01 times its factors), 8B Linear-layout layer at 16 tokens 170 -> 82 us, 8B x.u.v at 32
// tokens 114 -> 33 us.  What is left per launch is ~3.5-4.5 us of launch,
// ramp and in-block sums and 1.5 us (16 tokens) to 4 us (64) of slices.
// At 65-128 tokens two groups of 64 rows run side by side as blocks of their
// own, each streaming the weights (they meet in L2), so the time grows with
// the factors where the large tiles' is mostly fixed: decode_ok (api.hip) has
// the line between them.
#pragma once

#include "gemm_big.hpp"
#include "sync_area.hpp"

namespace svdmlp {

enum StreamW : int { SW_NATURAL = 0, SW_LINEAR = 1, SW_FP8 = 2 };

struct StreamSeg {
  const uint16_t* a;   // (T, K) bf16, row pitch K
  const void* w;       // (K, N), or (N, K) in the Linear layout
  const float* scale;  // per column (fp8), or null
  uint16_t* out;       // (T, N) bf16, row pitch ldo
  int64_t ldw;         // row pitch of w as stored (elements)
  int64_t ldo;         // row pitch of out (of out^T with out_t)
  int K, N;
  int ntiles;          // ceil(N / (128 cg))
  int ks;              // K per split, a multiple of 64
};

struct StreamParams {
  StreamSeg seg[2];       // DUAL: gate and up branch of one output (seg[0].out)
  int T, splits, tiles;   // tiles: column tiles over the segments (DUAL: of one)
  int groups;             // ceil(T / 64) groups of 64 token rows, each with units of its own
  int out_t;              // out is (N, T): T a multiple of 8
  float* slices;          // fp32, (tile, split, branch) slices of T x 128
  uint32_t slice_bytes;
  uint64_t* sync;         // tile counters (sync_area.hpp) and the timeout flag
  const uint16_t* resid;  // (T, N) added to bf16(out), row pitch ldo, or null
  int layer;              // a stage of the layer: NaN while the timeout flag is set
};

constexpr int kStRows = 64;  // token rows of a group
constexpr int kStMaxT = 2 * kStRows;
constexpr int kStThreads = 512;
constexpr int kGlMaxT = 2;  // tokens of the Linear GEMV stages (gemv_linear.hip)
constexpr int kStTileN = 128;
constexpr uint32_t kStNone = 0xfffffff0u;  // past the slice area: reads zeros

// Registers of one step: 32 H k of the tile's columns and the token rows.
template <int MT, int WK, int CG>
struct StStep {
  static constexpr bool B64 = WK == SW_FP8 && CG == 1;  // fp8 in 8-byte pieces
  // 32-k halves.  Linear: a lane reads 32 contiguous bytes of a row with two
  // loads, whose first touches every sector of the 16 rows' 128-byte lines
  static constexpr int H = WK == SW_LINEAR && MT <= 2 ? 2 : 1;
  u32x4 w[H][B64 ? 1 : 8];  // rows (natural, fp8) or columns (Linear)
  u32x2 w8[B64 ? 8 : 1];
  u32x4 a[H][MT];
};

// Two rows' 16-bit halves of one column: (lo of row 0, lo of row 1) or both highs.
__device__ __forceinline__ uint32_t st_pair(uint32_t r0, uint32_t r1, bool high) {
  return __builtin_amdgcn_perm(r1, r0, high ? 0x07060302u : 0x05040100u);
}

// Two of a dword's four fp8 e4m3fn values, widened exactly to bf16.
__device__ __forceinline__ uint32_t st_fp8_pair(uint32_t d, bool high) {
  return high ? __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d, 1.0f, true))
              : __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d, 1.0f, false));
}

// Issues the loads of the step at k0 (uniform) of a unit at columns n0.. of
// segment s; `live` false: nothing is fetched and every register is zero.
// Every lane's pieces lie inside the matrices or its offset lies past any
// buffer (K and N are multiples of 8, so a lane's 8 x 8 block is inside or
// outside as a whole): kOOB reads zeros whichever way the scalar offset
// enters the range check.
template <int MT, int WK, int CG>
__device__ __forceinline__ void st_load(const StreamSeg& s, const uint16_t* a, int T, int n0, int k0, bool live, int lr,
                                        int lg, StStep<MT, WK, CG>& r) {
  const int records = live ? 0x7ffffff0 : 0;
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a) + k0, 0, records, 0x00020000);
  constexpr int esz = WK == SW_FP8 ? 1 : 2;
  const char* wb = static_cast<const char*>(s.w) +
                   (WK == SW_LINEAR ? (int64_t)n0 * s.ldw + k0 : (int64_t)k0 * s.ldw + n0) * esz;
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(wb), 0, records, 0x00020000);
  const uint32_t ld = live ? (uint32_t)s.ldw * (uint32_t)esz : 0u;
  using S = StStep<MT, WK, CG>;
  // lane group lg, half h: k0 + 8 (H lg + h) .. + 7
  const uint32_t col_past = n0 + 8 * CG * lr < s.N ? 0u : kOOB;
  uint32_t k_past[S::H];
#pragma unroll
  for (int h = 0; h < S::H; ++h) k_past[h] = k0 + 8 * (S::H * lg + h) < s.K ? 0u : kOOB;
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int h = 0; h < S::H; ++h) {
      const uint32_t v = (WK == SW_LINEAR ? (uint32_t)(8 * lr) * ld + 16u * (uint32_t)(S::H * lg + h)
                                          : (uint32_t)(8 * (S::H * lg + h)) * ld + (uint32_t)(8 * CG * esz) * lr) |
                         col_past | k_past[h];
      if constexpr (S::B64)
        r.w8[j] = __builtin_amdgcn_raw_buffer_load_b64(rw, v, j * ld, 0);
      else
        r.w[h][j] = __builtin_amdgcn_raw_buffer_load_b128(rw, v, j * ld, 0);
    }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = 16 * mt + lr;
    const uint32_t row = m < T ? (uint32_t)m * (uint32_t)s.K * 2u : kOOB;
#pragma unroll
    for (int h = 0; h < S::H; ++h)
      r.a[h][mt] = __builtin_amdgcn_raw_buffer_load_b128(ra, (row + 16u * (uint32_t)(S::H * lg + h)) | k_past[h], 0, 0);
  }
}

// acc[g][mt][j]: columns 8 CG lr + 8 g + j of the tile.
template <int MT, int WK, int CG>
__device__ __forceinline__ void st_mul(const StStep<MT, WK, CG>& r, f32x4 (&acc)[CG][MT][8]) {
#pragma unroll
  for (int h = 0; h < StStep<MT, WK, CG>::H; ++h) {
#pragma unroll
  for (int p = 0; p < 4 * CG; ++p) {  // columns 2p and 2p + 1 of the lane's
    u32x4 fb[2];
    if constexpr (WK == SW_LINEAR) {
      fb[0] = r.w[h][2 * p];
      fb[1] = r.w[h][2 * p + 1];
    } else {
      uint32_t d[8];  // the pair of each row, as bf16
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if constexpr (WK == SW_NATURAL)
          d[j] = r.w[h][j][p];
        else if constexpr (CG == 1)
          d[j] = st_fp8_pair(r.w8[j][p >> 1], p & 1);
        else
          d[j] = st_fp8_pair(r.w[h][j][p >> 1], p & 1);
      }
#pragma unroll
      for (int e = 0; e < 2; ++e)
        fb[e] = u32x4{st_pair(d[0], d[1], e), st_pair(d[2], d[3], e), st_pair(d[4], d[5], e), st_pair(d[6], d[7], e)};
    }
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        acc[p / 4][mt][2 * (p % 4) + e] = mfma_chunk(r.a[h][mt], fb[e], acc[p / 4][mt][2 * (p % 4) + e], __bf16{});
  }
  }
}

template <int MT, int WK, int CG, bool DUAL>
__global__ __launch_bounds__(kStThreads, 2) void stream_kernel(StreamParams p) {
  constexpr int NWB = DUAL ? 4 : 8;  // waves per branch
  constexpr int BR = DUAL ? 2 : 1;
  __shared__ __attribute__((aligned(16))) float red[8][16 * kStTileN];
  __shared__ int last;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane & 15, lg = lane >> 4;
  const int m00 = blockIdx.y * kStRows;     // the group's first token row
  const int T = min(p.T - m00, kStRows);    // and its rows
  const uint32_t srows = min(p.T, kStRows);  // rows of a slice
  int splits = p.splits;
  asm volatile("" : "+s"(splits));  // loaded with the arguments above, not after the weights
  const int split = blockIdx.x / p.tiles;
  const int tile = blockIdx.x % p.tiles;
  const bool second = !DUAL && tile >= p.seg[0].ntiles;
  const StreamSeg& so = p.seg[second ? 1 : 0];                        // the output's segment
  const StreamSeg& s = p.seg[DUAL ? wave >> 2 : (second ? 1 : 0)];  // the segment this wave streams
  const int n0 = (second ? tile - p.seg[0].ntiles : tile) * kStTileN * CG;
  const int kb = split * s.ks, ke = min(s.K, kb + s.ks);
  const int wb = DUAL ? wave & 3 : wave;
  const uint16_t* const a = s.a + (int64_t)m00 * s.K;

  // A workspace whose persistent decode call timed out has tile counters in an
  // unknown state.  The layer then gives NaN until it is reset, as the
  // persistent layers do; the halves, which no wait precedes, run without the
  // counters: the first split's unit takes its tile's whole K.  The flag's load
  // is in flight with the weights' and looked at after them.
  const uint32_t flag = __hip_atomic_load(reinterpret_cast<uint32_t*>(&p.sync[kDlFlag]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  f32x4 acc[CG][MT][8];
#pragma unroll
  for (int g = 0; g < CG; ++g)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[g][mt][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // step i of this wave: part i % S of its (i / S)-th 64-k block
  constexpr int S = 2 / StStep<MT, WK, CG>::H;
  auto run = [&](int kb, int ke) {
    const int nblk = (ke - kb + 63) / 64;
    const int steps = nblk > wb ? (nblk - wb + NWB - 1) / NWB * S : 0;
    StStep<MT, WK, CG> r0, r1;
    auto load = [&](int i, StStep<MT, WK, CG>& r) {
      const int k = kb + 64 * (i / S * NWB + wb) + 32 * (i % S);
      st_load<MT, WK, CG>(s, a, T, n0, k, i < steps && k < ke, lr, lg, r);
    };
    load(0, r0);
    for (int i = 0; i < steps; i += 2) {
      load(i + 1, r1);
      __builtin_amdgcn_sched_barrier(0);
      st_mul<MT, WK, CG>(r0, acc);
      __builtin_amdgcn_sched_barrier(0);
      load(i + 2, r0);
      __builtin_amdgcn_sched_barrier(0);
      st_mul<MT, WK, CG>(r1, acc);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  run(kb, ke);
  if (splits > 1 && __builtin_amdgcn_readfirstlane(flag)) {
    if (split) return;
    run(ke, s.K);
    splits = 1;
  }

  const bool poison = flag != 0 && p.layer;

  // group g's column q of the tile (q = 8 lr + j)
  auto column = [&](int g, int q) { return CG == 1 ? q : (q >> 3) * (8 * CG) + 8 * g + (q & 7); };
  // tile value of token m, columns n .. n + 3 (v1: the up branch)
  auto finish = [&](int m, int n, f32x4 v0, f32x4 v1) -> u32x2 {
    const int col = n0 + n;
    if (so.scale) v0 *= *reinterpret_cast<const f32x4*>(so.scale + col);
    if constexpr (DUAL) {
      if (p.seg[1].scale) v1 *= *reinterpret_cast<const f32x4*>(p.seg[1].scale + col);
      v0 = f32x4{silu_f32(v0.x) * v1.x, silu_f32(v0.y) * v1.y, silu_f32(v0.z) * v1.z, silu_f32(v0.w) * v1.w};
    }
    u32x2 o = u32x2{pack_bf16x2(v0.x, v0.y), pack_bf16x2(v0.z, v0.w)};
    if (p.resid) {
      const u32x2 x = *reinterpret_cast<const u32x2*>(p.resid + (int64_t)(m00 + m) * so.ldo + col);
      o = u32x2{add_bf16x2(x.x, o.x), add_bf16x2(x.y, o.y)};
    }
    constexpr uint32_t kNaN2 = 0x7fc07fc0u;
    return poison ? u32x2{kNaN2, kNaN2} : o;
  };
  auto store = [&](int m, int n, u32x2 v) {
    *reinterpret_cast<u32x2*>(so.out + (int64_t)(m00 + m) * so.ldo + n0 + n) = v;
  };

  // ---- the 8 waves' sums, 16 token rows at a time: thread (row tid / 32,
  // columns 4 (tid % 32)..) adds them in wave order.  Lanes of the upper
  // eight column groups write their two 16-byte halves in the other order, so
  // that the lanes of a pass cover all 64 banks. ----
  const int qm = tid >> 5, qn = 4 * (tid & 31);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(p.slices, 0, (int)p.slice_bytes, 0x00020000);
  const int gtile = blockIdx.y * p.tiles + tile;  // the tile's counter
  const uint32_t unit = (uint32_t)(gtile * p.splits + split) * BR;
  const bool exchange = splits > 1 || p.out_t;
#pragma unroll
  for (int g = 0; g < CG; ++g) {
    const int n = column(g, qn);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if (16 * mt < T) {  // uniform
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const f32x4(&c)[8] = acc[g][mt];
          const f32x4 lo = f32x4{c[0][t], c[1][t], c[2][t], c[3][t]}, hi = f32x4{c[4][t], c[5][t], c[6][t], c[7][t]};
          const bool sw = lr & 8;
          float* d = &red[wave][(4 * lg + t) * kStTileN + 8 * lr];
          *reinterpret_cast<f32x4*>(d + (sw ? 4 : 0)) = sw ? hi : lo;
          *reinterpret_cast<f32x4*>(d + (sw ? 0 : 4)) = sw ? lo : hi;
        }
        __syncthreads();
        f32x4 v[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int w = 0; w < 8; ++w) v[w / NWB] += *reinterpret_cast<const f32x4*>(&red[w][qm * kStTileN + qn]);
        const int m = 16 * mt + qm;
        if (m < T && n0 + n < so.N) {
          if (!exchange) {
            store(m, n, finish(m, n, v[0], v[1]));
          } else {
#pragma unroll
            for (int b = 0; b < BR; ++b)
              __builtin_amdgcn_raw_buffer_store_b128(
                  u32x4{__float_as_uint(v[b].x), __float_as_uint(v[b].y), __float_as_uint(v[b].z), __float_as_uint(v[b].w)},
                  rs, ((unit + b) * CG * srows + (uint32_t)(g * T + m)) * (kStTileN * 4u) + 4u * (uint32_t)qn, 0, kDlSc1);
          }
        }
      }
    }
  }
  if (!exchange) return;

  // ---- K splits: the last unit of the tile to arrive sums the slices in
  // split order (the counter wraps to zero for the next launch) ----
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0)
    last = splits == 1 ||
           __builtin_amdgcn_atomic_inc32(dl_tile_counter(p.sync, gtile), (uint32_t)p.splits - 1u, __ATOMIC_RELAXED, "agent") ==
               (uint32_t)p.splits - 1u;
  __syncthreads();
  if (!last) return;
  uint16_t* const tl = reinterpret_cast<uint16_t*>(&red[0][0]);  // out_t: the tile as [column][token]
  const int tp = T + 8;
  const uint32_t unit0 = (uint32_t)(gtile * p.splits) * BR;
  constexpr int SB = DUAL ? 4 : 8;  // splits in flight
  for (int q = tid; q < T * 32 * CG; q += kStThreads) {  // (group, token, column quad), in slice order
    const int g = CG == 1 ? 0 : q / (T * 32), m = (q >> 5) - g * T, n = column(g, 4 * (q & 31));
    if (n0 + n >= so.N) continue;
    f32x4 v[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    for (int s0 = 0; s0 < splits; s0 += SB) {
      u32x4 x[SB][BR];
#pragma unroll
      for (int k = 0; k < SB; ++k)
#pragma unroll
        for (int b = 0; b < BR; ++b)
          x[k][b] = __builtin_amdgcn_raw_buffer_load_b128(
              rs, s0 + k < splits ? (unit0 + (uint32_t)((s0 + k) * BR + b)) * (srows * (uint32_t)(CG * kStTileN * 4)) + 16u * (uint32_t)q
                                    : kStNone,
              0, kDlSc1);
#pragma unroll
      for (int k = 0; k < SB; ++k)
#pragma unroll
        for (int b = 0; b < BR; ++b)
          v[b] += f32x4{__uint_as_float(x[k][b].x), __uint_as_float(x[k][b].y), __uint_as_float(x[k][b].z),
                        __uint_as_float(x[k][b].w)};
    }
    const u32x2 o = finish(m, n, v[0], v[1]);
    if (p.out_t) {
      tl[(n + 0) * tp + m] = (uint16_t)o.x;
      tl[(n + 1) * tp + m] = (uint16_t)(o.x >> 16);
      tl[(n + 2) * tp + m] = (uint16_t)o.y;
      tl[(n + 3) * tp + m] = (uint16_t)(o.y >> 16);
    } else {
      store(m, n, o);
    }
  }
  if (!p.out_t) return;
  __syncthreads();
  const int per = T / 8;
  for (int q = tid; q < kStTileN * CG * per; q += kStThreads) {
    const int n = q / per, i = q % per;
    if (n0 + n < so.N)
      *reinterpret_cast<u32x4*>(so.out + (int64_t)(n0 + n) * so.ldo + m00 + 8 * i) = *reinterpret_cast<const u32x4*>(tl + n * tp + 8 * i);
  }
}

}  // namespace svdmlp
