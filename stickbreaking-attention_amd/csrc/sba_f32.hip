// fp32 path: the same operator evaluated entirely in fp32, for fp32 inputs, on the fp32 matrix instruction
// (v_mfma_f32_32x32x2_f32: exact fp32 products and sums).
//
// What bounds it: the matrix pipe.  A 32x32x2 fp32 MFMA takes 64 cycles for 4096 FLOP, 1/16 of the bf16 rate, so a
// 32 x 32 block of (query, key) pairs costs 8192 (forward, D = 128), 12288 (dQ) or 16384 (dK/dV) matrix cycles against
// fewer than 2000 cycles of everything else.  Consequences for the design:
//   * no tile is shared between waves: an operand goes from global memory straight into the registers of the wave that
//     uses it (16 KB per 4096 cycles and wave, served by the L2), a phase ahead of its use, in the registers the phase
//     before has consumed.  One barrier per 128 keys; two waves per SIMD cover each other's element-wise math.
//   * the unit of work is small (32 query rows, or 32 keys, per workgroup of four waves), because the longest row
//     would otherwise be the critical path: a single wave needs 64 x 8192 cycles = 0.25 ms for 32 rows of 2048 keys,
//     twice what the whole chip needs for the rest of such a batch.  The four waves split the KEYS of the forward and
//     of dQ (sub-tiles of 32 dealt round robin, one scalar per row exchanged per step) and the ROWS of dK/dV (nothing
//     exchanged), and add their partial results through LDS at the end, in a fixed order: bit-reproducible.
// Measured: 12 heads x 128, 6143 tokens in sequences of up to 2048, forward + backward 0.99 ms; 86.7 ms on the vector ALU
// with one wave per query row and fp32 atomics for dK/dV.  32 heads x 2048 tokens: forward 0.34, dQ 0.49, dK/dV 0.67 ms =
// 100, 104 and 102 TFLOP/s of products, where a large fp32 matrix product reaches 154 on this chip.
//
//   fwd_f32_kernel     : keys swept in reverse from the diagonal (as sb_varlen_fwd.py:155-165), running product per row;
//                        records the product above every 32-key sub-tile in `carry`.
//   bwd_dq_f32_kernel  : keys swept forwards; A from the recorded products, g = A (dO.v - drem), C = prefix sum of g,
//                        dz = g - sigma C (sb_varlen_bwd.py:438-447), dQ += dZ K; records C below every sub-tile.
//   bwd_dkv_f32_kernel : key-stationary; dV += P^T dO, dK += dZ^T Q over the rows that see the keys.
//
// Register layout: S^T = K Q^T as in the 16-bit kernels (lane l owns query l%32 and the 16 consecutive keys
// 16*(l/32) + r).  The contraction index of an MFMA is split between the half-waves, k = l/32, and which element it
// stands for is free as long as both operands agree:
//   over head_dim : d = 8*i + 4*(l/32) + t for MFMA 4*i + t, so a lane reads 16-byte pieces of its row from LDS;
//   over keys/rows: index 16*(l/32) + r for MFMA r: the score registers are the A operand as they stand.
#include "sba_device.hpp"
#include "sba_host.hpp"
#include "sba_params.hpp"
#include "sba_sched.hpp"

#include <type_traits>

namespace sba {

constexpr int kF32Rows = 32;                       // query rows, or keys, per workgroup
constexpr int kF32Split = kBlockQ / kF32Rows;      // workgroups per 128-row query tile of the schedule
constexpr int kF32KeySplit = kBlockK / kF32Rows;   // workgroups per 64-key tile of the schedule
constexpr int kF32TrStride = 36;                   // floats per row of the transposition buffers

enum : int { kF32Padded = 0, kF32Exact = 1, kF32Far = 2 };      // how rows are read, see Operand

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int r = 0; r < 16; r++) z[r] = 0.f;
  return z;
}
typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4_u;      // rows need only be 4-byte aligned

// 32 consecutive rows of a [.., token, head_dim] tensor as the source of one operand.  A raw buffer resource per 32 rows:
// rows at or beyond `last + 1` read as zero, and offsets stay small whatever the length of the sequence.
// (Rows more than 2^24 elements apart, of which 32 span more than 32-bit offsets reach, are read through pointers: `p`.)
struct Rows32 {
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t stride_bytes;
  const float* p;
  int64_t stride;
  int n;
};
__device__ __forceinline__ Rows32 rows32(const float* base, int64_t stride, int first, int rows_total, int D) {
  Rows32 r;
  r.stride_bytes = (uint32_t)stride * 4u;
  const int n = min(rows_total - first, 32);
  const float* p = base + (int64_t)first * stride;
  r.p = p; r.stride = stride; r.n = n;
  r.rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, n > 0 ? (int)((uint32_t)(n - 1) * r.stride_bytes + 4u * (uint32_t)D) : 0, 0x00020000);
  return r;
}

// An operand is 32 rows in DH/2 registers per lane, in parts of C columns (64 or 32): part p holds, of rows 16*half + r, the
// columns p*C + NC*(l%32) + j, NC = C/32, in register (p*16 + r)*NC + j.  That is the B operand of a contraction over the
// rows as it stands, and 64 lanes read two runs of C*4 contiguous bytes per instruction.  (A lane per row, what a
// contraction over head_dim wants, costs a cache access per lane when loaded like that: measured 1024 instead of 290 per
// 32 x 128 operand, and the kernels were bound by them.  Those operands go through LDS, a part at a time.)
// kF32Exact: head_dim == DH.  kF32Padded: an element beyond head_dim is asked for outside the buffer and reads as zero.
// kF32Far: any head_dim, rows at any distance.
template <int DH> struct Parts {
  static constexpr int C = DH == 128 ? 64 : 32, N = DH / C, NC = C / 32;
  static constexpr int kTurn = 32 * (C + 4);      // floats of a wave's scratch: [32 rows][C + 4]
};
template <int DH> __device__ __forceinline__ int out_col(int dt, int col) {
  typedef Parts<DH> P;
  return (dt / P::NC) * P::C + P::NC * col + dt % P::NC;
}
template <int DH, int kMode>
struct Operand {
  typedef Parts<DH> P;
  Rows32 src;
  uint32_t voff;      // 16 * half rows, this lane's first column
  int col, D, half16;
  __device__ __forceinline__ void fill_piece(float (&x)[DH / 2], int part, int r) const {
    const uint32_t soff = (uint32_t)r * src.stride_bytes;
    float* y = x + (part * 16 + r) * P::NC;
    if (kMode == kF32Exact && P::NC == 2) {
      const f32x2 v = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(src.rsrc, voff + 4 * part * P::C, soff, 0));
      y[0] = v[0]; y[P::NC - 1] = v[1];
    } else if (kMode == kF32Far) {
      const int row = half16 + r, d = part * P::C + P::NC * col;
#pragma unroll
      for (int j = 0; j < P::NC; j++) y[j] = row < src.n && d + j < D ? src.p[row * src.stride + d + j] : 0.f;
    } else {
#pragma unroll
      for (int j = 0; j < P::NC; j++) {
        const uint32_t vo = kMode == kF32Exact || part * P::C + P::NC * col + j < D ? voff + 4 * (part * P::C + j) : (uint32_t)kOutside;
        y[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(src.rsrc, vo, soff, 0));
      }
    }
  }
  __device__ __forceinline__ void fill_part(float (&x)[DH / 2], int part) const {
#pragma unroll
    for (int r = 0; r < 16; r++) fill_piece(x, part, r);
  }
  __device__ __forceinline__ void fill(float (&x)[DH / 2]) const {
#pragma unroll
    for (int part = 0; part < P::N; part++) fill_part(x, part);
  }
};
template <int DH, int kMode>
__device__ __forceinline__ Operand<DH, kMode> operand(const float* base, int64_t stride, int first, int rows_total, int half, int col, int D) {
  const Rows32 s = rows32(base, stride, first, rows_total, D);
  return Operand<DH, kMode>{s, 16u * (uint32_t)half * s.stride_bytes + 4u * (uint32_t)out_col<DH>(0, col), col, D, 16 * half};
}

// The phases.  Each consumes what x holds, part by part, and refills a part's registers for the phase that follows once
// they are free.  The refilling loads are dealt among the MFMAs: a load takes the memory pipe 13 cycles, and four waves
// that issue 16 of them back to back stand still for 850 (measured); behind an MFMA each the wait is hidden.  The last
// part a contraction consumes is refilled among the first MFMAs of the next phase: that phase is told so (`late`).

// acc = (rows in x) . (rows in LDS, stride DH + 4), contracted over head_dim; row `xrow` of x and the LDS row `lds_row`
// are this lane's.  kLdsIsA: the LDS rows are the A operand (output rows).  x goes through the wave's scratch; the
// operands of four MFMAs are read one group ahead.
template <int DH, int kMode, bool kLdsIsA>
__device__ __forceinline__ f32x16 score_phase(float (&x)[DH / 2], float* turn, int xrow, const float* lds_row, int half, int col,
                                              const Operand<DH, kMode>& next, const Operand<DH, kMode>& late, bool has_late) {
  typedef Parts<DH> P;
  constexpr int S = P::C + 4, G = P::C / 8;      // groups of four MFMAs per part
  f32x16 acc = zero16();
#pragma unroll
  for (int part = 0; part < P::N; part++) {
    __builtin_amdgcn_sched_barrier(0);
    const float* yr = lds_row + part * P::C + 4 * half;
    const float* xr = turn + xrow * S + 4 * half;
    f32x4 b = *reinterpret_cast<const f32x4*>(yr);
#pragma unroll
    for (int r = 0; r < 16; r++)
#pragma unroll
      for (int j = 0; j < P::NC; j++) turn[(16 * half + r) * S + P::NC * col + j] = x[(part * 16 + r) * P::NC + j];
    f32x4 a = *reinterpret_cast<const f32x4*>(xr);
    auto segment = [&](auto with_late) {
#pragma unroll
      for (int i = 0; i < G; i++) {
        f32x4 an = a, bn = b;
        __builtin_amdgcn_sched_barrier(0);
        if (i + 1 < G) {
          an = *reinterpret_cast<const f32x4*>(xr + 8 * (i + 1));
          bn = *reinterpret_cast<const f32x4*>(yr + 8 * (i + 1));
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
          __builtin_amdgcn_sched_barrier(0);
          acc = kLdsIsA ? mfma_f32(b[t], a[t], acc) : mfma_f32(a[t], b[t], acc);
          __builtin_amdgcn_sched_barrier(0);
          constexpr int kM = 4 * G;                          // MFMAs of the segment
          const int m = 4 * i + t;
          // (the late part is wanted first: its loads go ahead of the others)
          if (decltype(with_late)::value) {
#pragma unroll
            for (int r = 0; r < 32; r++)
              if (r * kM / 32 == m) { if (r < 16) late.fill_piece(x, P::N - 1, r); else next.fill_piece(x, part, r - 16); }
          } else {
#pragma unroll
            for (int r = 0; r < 16; r++)
              if (r * kM / 16 == m) next.fill_piece(x, part, r);
          }
        }
        a = an; b = bn;
      }
    };
    if (part == 0 && P::N > 1 && has_late) segment(std::true_type{}); else segment(std::false_type{});
  }
  __builtin_amdgcn_sched_barrier(0);
  return acc;
}

// acc[dt] += a . x, contraction over 32 rows.
template <int DH, int kMode>
__device__ __forceinline__ void contract_phase(f32x16 (&acc)[DH / 32], const float (&a)[16], float (&x)[DH / 2],
                                               const Operand<DH, kMode>& next, bool refill, const Operand<DH, kMode>& late,
                                               bool has_late) {
  typedef Parts<DH> P;
#pragma unroll
  for (int part = 0; part < P::N; part++) {
#pragma unroll
    for (int r = 0; r < 16; r++) {
#pragma unroll
      for (int j = 0; j < P::NC; j++) {
        __builtin_amdgcn_sched_barrier(0);
        acc[part * P::NC + j] = mfma_f32(a[r], x[(part * 16 + r) * P::NC + j], acc[part * P::NC + j]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (part > 0) { if (refill) next.fill_piece(x, part - 1, r); }
      else if (P::N > 1 && has_late) late.fill_piece(x, P::N - 1, r);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  if (P::N == 1 && refill) next.fill(x);
}

// 32 rows into LDS, [row][DH + 4] floats, zeros beyond the last row and beyond head_dim; all threads take part.
template <int DH, int kMode>
__device__ __forceinline__ void stage_rows(float* lds, const Rows32& s, int D) {
  if (kMode == kF32Exact) {
#pragma unroll
    for (int i = 0; i < 32 * (DH / 4) / kThreads; i++) {
      const int idx = threadIdx.x + kThreads * i, row = idx / (DH / 4), d = (idx % (DH / 4)) * 4;
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(s.rsrc, (uint32_t)row * s.stride_bytes + 4 * d, 0, 0);
      *reinterpret_cast<u32x4*>(lds + row * (DH + 4) + d) = v;
    }
  } else if (kMode == kF32Far) {
    for (int idx = threadIdx.x; idx < 32 * DH; idx += kThreads) {
      const int row = idx / DH, d = idx % DH;
      lds[row * (DH + 4) + d] = row < s.n && d < D ? s.p[row * s.stride + d] : 0.f;
    }
  } else {
    for (int idx = threadIdx.x; idx < 32 * DH; idx += kThreads) {
      const int row = idx / DH, d = idx % DH;
      const uint32_t v = __builtin_amdgcn_raw_buffer_load_b32(s.rsrc, d < D ? (uint32_t)row * s.stride_bytes + 4 * d : (uint32_t)kOutside, 0, 0);
      lds[row * (DH + 4) + d] = __builtin_bit_cast(float, v);
    }
  }
}

// 1/x for 1 <= x <= 2^101: the hardware's reciprocal (1 ulp) and one Newton step.
__device__ __forceinline__ float rcp_f32(float x) {
  const float y = fast_rcp(x);
  return fmaf(y, fmaf(-x, y, 1.f), y);
}

// Sticks of this lane's 16 keys, swept from the highest down: sigma in `beta`, the product of (1 - sigma) over the
// lane's higher keys in `pe`; returns the product over all 16.  Key R is visible iff R < lim.
// The hardware's exponential flushes results below 2^-126; a wave that holds such a logit takes the library's, which does not
// and gives the same bits elsewhere (5 instructions more per key: taken always, 12 heads x 6 x 1024 x 128, forward and
// backward, 970 -> 996 us; taken so, 970).  sigma is the quotient e / (1 + e) with its rounding error taken out, not a multiple
// of the rounded reciprocal, which takes 2 to 5 % off the error of every output.  Both together cost 0.9 % of a pass at head_dim 128,
// 1.8 % at 64 and 96 and 2.7 % at 32 (12 heads, 6143 tokens: 980 -> 989, 515 -> 525, 740 -> 753, 298 -> 307 us).
__device__ __forceinline__ float sticks_f32(const f32x16& s, float scale_log2, int lim, float (&beta)[16], float (&pe)[16]) {
  float x[16], lowest = 0.f;
#pragma unroll
  for (int R = 0; R < 16; R++) {
    x[R] = fminf(s[R] * scale_log2, 100.f);
    lowest = fminf(lowest, x[R]);
  }
  if (__any(lowest < -126.f)) {
#pragma unroll
    for (int R = 0; R < 16; R++) x[R] = exp2f(x[R]);
  } else {
#pragma unroll
    for (int R = 0; R < 16; R++) x[R] = fast_exp2(x[R]);
  }
  float run = 1.f;
#pragma unroll
  for (int R = 15; R >= 0; --R) {
    const float e = R < lim ? x[R] : 0.f, one_e = 1.f + e;
    const float omb = rcp_f32(one_e), b = e * omb;
    beta[R] = fmaf(fmaf(-one_e, b, e), omb, b);
    pe[R] = run;
    run *= omb;
  }
  return run;
}

// Sum the four waves' partial [32 rows][DH] results through LDS and store them (times `scale`, plus add_scale[row] *
// add[row] when `add` is given).  acc[dt][r]: row 8*(r/4) + 4*half + r%4, column out_col(dt).  All waves take part.
template <int DH, int kMode>
__device__ __forceinline__ void reduce_store_f32(float* lds, const f32x16 (&acc)[DH / 32], float scale, float* out, int64_t stride,
                                                 int rows, int D, const float* add = nullptr, int64_t add_stride = 0,
                                                 const float* add_scale = nullptr) {
  constexpr int NB = DH / 32, kStride = DH + 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, half = lane >> 5, col = lane & 31;
  __syncthreads();
  float* mine = lds + wave * 32 * kStride;
#pragma unroll
  for (int r = 0; r < 16; r++)
#pragma unroll
    for (int dt = 0; dt < NB; dt++)
      mine[(8 * (r >> 2) + 4 * half + (r & 3)) * kStride + out_col<DH>(dt, col)] = acc[dt][r];
  __syncthreads();
  for (int idx = threadIdx.x; idx < 32 * (DH / 4); idx += kThreads) {
    const int row = idx / (DH / 4), d0 = (idx % (DH / 4)) * 4;
    if (row >= rows || d0 >= D) continue;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kWaves; w++) v += *reinterpret_cast<const f32x4*>(lds + (w * 32 + row) * kStride + d0);
    v *= scale;
    float* o = out + (int64_t)row * stride + d0;
    const float* a = add ? add + (int64_t)row * add_stride + d0 : nullptr;
    const float as = add ? add_scale[row] : 0.f;
    if (kMode == kF32Exact) {
      if (a) { const f32x4_u w = *reinterpret_cast<const f32x4_u*>(a); v += as * (f32x4){w[0], w[1], w[2], w[3]}; }
      *reinterpret_cast<f32x4_u*>(o) = f32x4_u{v[0], v[1], v[2], v[3]};
    } else {
#pragma unroll
      for (int t = 0; t < 4; t++)
        if (d0 + t < D) o[t] = v[t] + (a ? as * a[t] : 0.f);
    }
  }
}

// LDS of the row-stationary kernels: kTiles tiles of 32 rows and the waves' scratch; the final sums lie over both.
template <int DH, int kTiles>
struct RowsF32Lds {
  static constexpr int kLoop = kTiles * 32 * (DH + 4) + kWaves * Parts<DH>::kTurn, kRed = kWaves * 32 * (DH + 4);
  static constexpr int kFloats = kLoop > kRed ? kLoop : kRed;
};

// (Width 96 keeps three waves per SIMD by spilling four registers; 177 registers and two waves take 4 % of a pass more.)
template <int DH, int kMode>
__global__ __launch_bounds__(kThreads, DH == 96 ? 3 : 2) void fwd_f32_kernel(FwdParams p) {
  constexpr int NB = DH / 32;
  __shared__ __attribute__((aligned(16))) float lds[RowsF32Lds<DH, 1>::kFloats];      // Q rows and the waves' scratch, then the final sums
  __shared__ float xch[2][kWaves][32];
  __shared__ float rem_lds[32];
  if ((int)blockIdx.x < p.sched.service) {
    forward_service(p.sched, blockIdx.x);
    return;
  }
  const int wg = blockIdx.x - p.sched.service;
  int head, slot, sub;
  xcd_head_tile_sub(wg, kF32Split, p.num_heads, &head, &slot, &sub);
  Tile tile;
  int64_t r0, r1;
  if (!forward_tile(p, slot, sub, kF32Rows, &tile, &r0, &r1)) {
    if (r0 < r1) {
      zero_rows<float>(p.o, head, r0, r1, p.head_dim);      // rows of no sequence: o = rem = 0
      for (int64_t r = r0 + threadIdx.x; r < r1; r += kThreads) {
        ((float*)p.rem.ptr)[head * p.rem.sh + r * p.rem.st] = 0.f;
        p.row_stat[head * p.stat_sh + r] = 0.f;
      }
    }
    return;
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, col = lane & 31;
  const int L = tile.seq_len, ac = p.attend_current, D = p.head_dim;
  const int q0 = tile.origin + sub * kF32Rows;
  if (q0 >= L) return;
  const int64_t tok0 = tile.seq_start;
  const float* qb = (const float*)p.q.ptr + tile.seq_id * p.q.sb + head * p.q.sh + tok0 * p.q.st;
  const float* kb = (const float*)p.k.ptr + tile.seq_id * p.k.sb + head * p.k.sh + tok0 * p.k.st;
  const float* vb = (const float*)p.v.ptr + tile.seq_id * p.v.sb + head * p.v.sh + tok0 * p.v.st;
  const int64_t n_qt = (L + kBlockQ - 1) / kBlockQ;
  float* carry = p.carry ? p.carry + (int64_t)head * p.carry_head_stride + tile.carry_base : nullptr;

  const int qi = q0 + col;
  const int last_key = min(q0 + kF32Rows, L) - 2 + ac;
  const int n_sub = last_key < 0 ? 0 : last_key / 32 + 1, n_steps = (n_sub + kWaves - 1) / kWaves;
  const int krow = mfma_row_to_key32(col);
  auto k_of = [&](int u) { return operand<DH, kMode>(kb, p.k.st, 32 * u, L, half, col, D); };
  auto v_of = [&](int u) { return operand<DH, kMode>(vb, p.v.st, 32 * u, L, half, col, D); };
  float x[DH / 2];
  // Wave w takes sub-tile n_sub - 1 - (4 t + w) in step t.
  int U = n_sub - 1 - wave;
  if (U >= 0) k_of(U).fill(x);
  stage_rows<DH, kMode>(lds, rows32(qb, p.q.st, q0, L, D), D);
  const float* q_lds = lds + col * (DH + 4);
  float* turn = lds + 32 * (DH + 4) + wave * Parts<DH>::kTurn;
  f32x16 oacc[NB];
#pragma unroll
  for (int dt = 0; dt < NB; dt++) oacc[dt] = zero16();
  float prod = 1.f;      // product over the keys of the steps done so far
  __syncthreads();
  for (int t = 0; t < n_steps; ++t, U -= kWaves) {
    float beta[16], pe[16];
    float run = 1.f, oth = 1.f;
    if (U >= 0) {
      const f32x16 s = score_phase<DH, kMode, false>(x, turn, krow, q_lds, half, col, v_of(U), k_of(U), t > 0);
      run = sticks_f32(s, p.scale_log2, qi + ac - 32 * U - 16 * half, beta, pe);
      oth = other_half(run, half);
    }
    if (half == 0) xch[t & 1][wave][col] = run * oth;
    lds_barrier();
    float above = prod;
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
      const float y = xch[t & 1][w][col];
      if (w < wave) above *= y;
      prod *= y;
    }
    if (U >= 0) {
      if (carry && half == 0) carry[carry_offset(U, n_qt) + (qi - kBlockQ * (U >> 2))] = above;
      const float seed = half ? above : above * oth;        // the upper half-wave holds the higher keys
#pragma unroll
      for (int r = 0; r < 16; r++) pe[r] = beta[r] * (pe[r] * seed);
      contract_phase<DH, kMode>(oacc, pe, x, k_of(U - kWaves), U >= kWaves, k_of(U), false);
    }
  }
  if (wave == 0 && half == 0) {
    rem_lds[col] = prod;
    if (qi < L) {
      ((float*)p.rem.ptr)[tile.seq_id * p.rem.sb + head * p.rem.sh + (tok0 + qi) * p.rem.st] = prod;
      p.row_stat[tile.seq_id * p.stat_sb + head * p.stat_sh + tok0 + qi] = log2f(prod);
    }
  }
  float* ob = (float*)p.o.ptr + tile.seq_id * p.o.sb + head * p.o.sh + (tok0 + q0) * p.o.st;
  reduce_store_f32<DH, kMode>(lds, oacc, 1.f, ob, p.o.st, L - q0, D, p.add_rem ? vb + (int64_t)q0 * p.v.st : nullptr, p.v.st, rem_lds);
}

template <int DH, int kMode>
__global__ __launch_bounds__(kThreads, 2) void bwd_dq_f32_kernel(BwdParams p) {
  constexpr int NB = DH / 32;
  __shared__ __attribute__((aligned(16))) float lds[RowsF32Lds<DH, 2>::kFloats];      // Q and dO rows and the waves' scratch, then the final sums
  __shared__ float xch[2][kWaves][32];
  int head, slot, sub;
  xcd_head_tile_sub(blockIdx.x, kF32Split, p.num_heads, &head, &slot, &sub);
  if (slot >= p.counts[kCountQ]) {
    int64_t r0, r1;
    if (uncovered_rows(p.counts, slot, p.total_tokens, sub, kF32Rows, &r0, &r1)) {      // rows of no sequence: zero gradients
      zero_rows<float>(p.dq, head, r0, r1, p.head_dim);
      zero_rows<float>(p.dk, head, r0, r1, p.head_dim);
      zero_rows<float>(p.dv, head, r0, r1, p.head_dim);
    }
    return;
  }
  const Tile tile = p.q_tiles[slot];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, col = lane & 31;
  const int L = tile.seq_len, ac = p.attend_current, D = p.head_dim;
  const int q0 = tile.origin + sub * kF32Rows;
  if (q0 >= L) return;
  const int64_t tok0 = tile.seq_start;
  const float* qb = (const float*)p.q.ptr + tile.seq_id * p.q.sb + head * p.q.sh + tok0 * p.q.st;
  const float* kb = (const float*)p.k.ptr + tile.seq_id * p.k.sb + head * p.k.sh + tok0 * p.k.st;
  const float* vb = (const float*)p.v.ptr + tile.seq_id * p.v.sb + head * p.v.sh + tok0 * p.v.st;
  const float* dob = (const float*)p.d_o.ptr + tile.seq_id * p.d_o.sb + head * p.d_o.sh + tok0 * p.d_o.st;
  const int64_t n_qt = (L + kBlockQ - 1) / kBlockQ;
  const int64_t slot0 = (int64_t)head * p.carry_head_stride + tile.carry_base;
  const float* carry = p.carry + slot0;
  float* prefix_out = p.prefix + slot0;

  const int qi = q0 + col;
  const int last_key = min(q0 + kF32Rows, L) - 2 + ac;
  const int n_sub = last_key < 0 ? 0 : last_key / 32 + 1, n_steps = (n_sub + kWaves - 1) / kWaves;
  const int krow = mfma_row_to_key32(col);
  auto k_of = [&](int u) { return operand<DH, kMode>(kb, p.k.st, 32 * u, L, half, col, D); };
  auto v_of = [&](int u) { return operand<DH, kMode>(vb, p.v.st, 32 * u, L, half, col, D); };
  float x[DH / 2];
  int U = wave;            // wave w takes sub-tile 4 t + w in step t
  if (U < n_sub) k_of(U).fill(x);
  stage_rows<DH, kMode>(lds, rows32(qb, p.q.st, q0, L, D), D);
  stage_rows<DH, kMode>(lds + 32 * (DH + 4), rows32(dob, p.d_o.st, q0, L, D), D);
  const float* q_lds = lds + col * (DH + 4);
  const float* do_lds = q_lds + 32 * (DH + 4);
  float* turn = lds + 64 * (DH + 4) + wave * Parts<DH>::kTurn;
  float drem = 0.f;
  if (qi < L && p.d_rem.ptr) drem = ((const float*)p.d_rem.ptr)[tile.seq_id * p.d_rem.sb + head * p.d_rem.sh + (tok0 + qi) * p.d_rem.st];
  __syncthreads();
  if (p.add_rem) {
    // The forward wrote o + rem * v: the gradient reaching rem is d_rem + d_o . v_i.
    const float* vi = vb + (int64_t)min(qi, L - 1) * p.v.st;
    float dot = 0.f;
    for (int d = half; d < D; d += 2) dot = fmaf(lds[(32 + col) * (DH + 4) + d], vi[d], dot);
    drem += dot + other_half(dot, half);
  }
  if (wave == 0 && half == 0 && qi < L) p.drem_eff[tile.seq_id * p.drem_sb + head * p.stat_sh + tok0 + qi] = drem;

  f32x16 dqacc[NB];
#pragma unroll
  for (int dt = 0; dt < NB; dt++) dqacc[dt] = zero16();
  float prefix = 0.f;      // sum of g over the keys of the steps done so far
  for (int t = 0; t < n_steps; ++t, U += kWaves) {
    float beta[16], dz[16];
    float tot = 0.f, fix = 0.f;
    const int64_t cslot = carry_offset(U, n_qt) + (qi - kBlockQ * (U >> 2));
    const bool active = U < n_sub;
    if (active) {
      const float prod_in = carry[cslot];
      const f32x16 s = score_phase<DH, kMode, false>(x, turn, krow, q_lds, half, col, v_of(U), k_of(U), t > 0);
      const f32x16 dp = score_phase<DH, kMode, false>(x, turn, krow, do_lds, half, col, k_of(U), k_of(U), false);
      float pe[16];
      const float run = sticks_f32(s, p.scale_log2, qi < L ? qi + ac - 32 * U - 16 * half : 0, beta, pe);
      const float oth = other_half(run, half);
      const float seed = half ? prod_in : prod_in * oth;
      float acc = 0.f;
#pragma unroll
      for (int R = 0; R < 16; R++) {
        const float g = beta[R] * (pe[R] * seed) * (dp[R] - drem);
        acc += g;
        dz[R] = g - beta[R] * acc;
      }
      const float oth_g = other_half(acc, half);
      tot = acc + oth_g;
      fix = half ? oth_g : 0.f;                              // the lower half-wave holds the lower keys
    }
    if (half == 0) xch[t & 1][wave][col] = tot;
    lds_barrier();
    float below = prefix;
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
      const float y = xch[t & 1][w][col];
      if (w < wave) below += y;
      prefix += y;
    }
    if (active) {
      if (half == 0) prefix_out[cslot] = below;
      const float fixup = below + fix;
#pragma unroll
      for (int r = 0; r < 16; r++) dz[r] -= beta[r] * fixup;
      contract_phase<DH, kMode>(dqacc, dz, x, k_of(U + kWaves), U + kWaves < n_sub, k_of(U), false);
    }
  }
  float* dqb = (float*)p.dq.ptr + tile.seq_id * p.dq.sb + head * p.dq.sh + (tok0 + q0) * p.dq.st;
  reduce_store_f32<DH, kMode>(lds, dqacc, p.logit_scale, dqb, p.dq.st, L - q0, D);
}

template <int DH>
struct DkvF32Lds {
  static constexpr int kRowStride = DH + 4;
  static constexpr int kK = 0, kV = kK + 32 * kRowStride;                             // the workgroup's keys
  static constexpr int kTr = kV + 32 * kRowStride;                                    // per wave: operand scratch; P^T, dZ^T
  static constexpr int kTrWave = Parts<DH>::kTurn > 2 * 32 * kF32TrStride ? Parts<DH>::kTurn : 2 * 32 * kF32TrStride;
  static constexpr int kLoop = kTr + kWaves * kTrWave;
  static constexpr int kRed = kWaves * 32 * kRowStride;                               // final sums, over the above
  static constexpr int kFloats = (kLoop > kRed ? kLoop : kRed) + 32;                  // + rem of 32 rows
};

template <int DH, int kMode>
__global__ __launch_bounds__(kThreads, 2) void bwd_dkv_f32_kernel(BwdParams p) {
  constexpr int NB = DH / 32;
  typedef DkvF32Lds<DH> Lds;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  int head, slot, sub;
  xcd_head_tile_sub(blockIdx.x, kF32KeySplit, p.num_heads, &head, &slot, &sub);
  if (slot >= p.counts[kCountK]) return;
  const Tile tile = p.k_tiles[slot];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, col = lane & 31;
  const int L = tile.seq_len, ac = p.attend_current, D = p.head_dim;
  const int k0 = tile.origin + sub * kF32Rows;
  if (k0 >= L) return;
  const int64_t tok0 = tile.seq_start;
  const float* qb = (const float*)p.q.ptr + tile.seq_id * p.q.sb + head * p.q.sh + tok0 * p.q.st;
  const float* kb = (const float*)p.k.ptr + tile.seq_id * p.k.sb + head * p.k.sh + tok0 * p.k.st;
  const float* vb = (const float*)p.v.ptr + tile.seq_id * p.v.sb + head * p.v.sh + tok0 * p.v.st;
  const float* dob = (const float*)p.d_o.ptr + tile.seq_id * p.d_o.sb + head * p.d_o.sh + tok0 * p.d_o.st;
  const int64_t n_qt = (L + kBlockQ - 1) / kBlockQ;
  const int U = k0 >> 5;
  const int64_t slot0 = (int64_t)head * p.carry_head_stride + tile.carry_base + carry_offset(U, n_qt) - kBlockQ * (U >> 2);
  const float* carry = p.carry + slot0;
  const float* prefix = p.prefix + slot0;
  const float* drem_plane = p.drem_eff + tile.seq_id * p.drem_sb + head * p.stat_sh + tok0;

  auto q_of = [&](int b) { return operand<DH, kMode>(qb, p.q.st, 32 * b, L, half, col, D); };
  auto do_of = [&](int b) { return operand<DH, kMode>(dob, p.d_o.st, 32 * b, L, half, col, D); };
  // Row blocks of 32 that see these keys: from the last one down to the one that holds the keys' own rows; wave w takes every
  // fourth.  (Downwards the loop needs one bound fewer in registers: 20 instead of 64 of them spilled at head_dim 128, 2 % of
  // the pass.)
  const int nb = k0 + 1 - ac < L ? (L + 31) / 32 : 0;
  int b = nb - 1 - wave;
  float x[DH / 2];
  if (b >= U) q_of(b).fill(x);
  // K and V of the 32 keys stay in LDS for the A operands of S^T and dP^T.
  stage_rows<DH, kMode>(lds + Lds::kK, rows32(kb, p.k.st, k0, L, D), D);
  stage_rows<DH, kMode>(lds + Lds::kV, rows32(vb, p.v.st, k0, L, D), D);
  const int krow = mfma_row_to_key32(col);
  const float* k_lds = lds + Lds::kK + krow * Lds::kRowStride;
  const float* v_lds = lds + Lds::kV + krow * Lds::kRowStride;
  float* turn = lds + Lds::kTr + wave * Lds::kTrWave;
  float* tp = turn;                                        // P^T [key][row], then dZ^T
  float* tz = tp + 32 * kF32TrStride;

  f32x16 dkacc[NB], dvacc[NB];
#pragma unroll
  for (int dt = 0; dt < NB; dt++) { dkacc[dt] = zero16(); dvacc[dt] = zero16(); }
  __syncthreads();
  for (; b >= U; b -= kWaves) {
    const int qi = 32 * b + col;
    const bool row_ok = qi < L;
    const float prod_in = carry[qi], prefix_in = prefix[qi];
    const float drem = row_ok ? drem_plane[qi] : 0.f;
    const f32x16 s = score_phase<DH, kMode, true>(x, turn, col, k_lds, half, col, do_of(b), q_of(b), b < nb - kWaves);
    const f32x16 dp = score_phase<DH, kMode, true>(x, turn, col, v_lds, half, col, do_of(b), do_of(b), false);
    {
      float beta[16], pe[16];
      const float run = sticks_f32(s, p.scale_log2, row_ok ? qi + ac - k0 - 16 * half : 0, beta, pe);
      const float oth = other_half(run, half);
      const float seed = half ? prod_in : prod_in * oth;
      // To [key][row] order (wave-private): the contraction over rows needs a lane per key.
      float acc = 0.f;
#pragma unroll
      for (int R = 0; R < 16; R++) {
        const float a = beta[R] * (pe[R] * seed);
        const float g = a * (dp[R] - drem);
        tp[(16 * half + R) * kF32TrStride + col] = a;
        acc += g;
        pe[R] = g - beta[R] * acc;
      }
      const float oth_g = other_half(acc, half);
      const float fixup = prefix_in + (half ? oth_g : 0.f);
#pragma unroll
      for (int R = 0; R < 16; R++) tz[(16 * half + R) * kF32TrStride + col] = pe[R] - beta[R] * fixup;
    }
    auto transposed = [&](const float* t, float (&y)[16]) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(t + col * kF32TrStride + 16 * half + 4 * i);
#pragma unroll
        for (int k = 0; k < 4; k++) y[4 * i + k] = v[k];
      }
    };
    float y[16];
    transposed(tp, y);
    contract_phase<DH, kMode>(dvacc, y, x, q_of(b), true, q_of(b), false);
    transposed(tz, y);
    contract_phase<DH, kMode>(dkacc, y, x, q_of(b - kWaves), b - kWaves >= U, q_of(b), true);
  }
  float* rem_lds = lds + Lds::kFloats - 32;
  if (p.add_rem && threadIdx.x < 32 && k0 + (int)threadIdx.x < L)      // the forward wrote o + rem * v: dv_i gains rem_i * d_o_i
    rem_lds[threadIdx.x] = exp2f(p.row_stat[tile.seq_id * p.stat_sb + head * p.stat_sh + tok0 + k0 + threadIdx.x]);
  float* dvb = (float*)p.dv.ptr + tile.seq_id * p.dv.sb + head * p.dv.sh + (tok0 + k0) * p.dv.st;
  float* dkb = (float*)p.dk.ptr + tile.seq_id * p.dk.sb + head * p.dk.sh + (tok0 + k0) * p.dk.st;
  reduce_store_f32<DH, kMode>(lds, dvacc, 1.f, dvb, p.dv.st, L - k0, D, p.add_rem ? dob + (int64_t)k0 * p.d_o.st : nullptr,
                               p.d_o.st, rem_lds);
  reduce_store_f32<DH, kMode>(lds, dkacc, p.logit_scale, dkb, p.dk.st, L - k0, D);
}

// head_dim is rounded up to a multiple of 32 (the matrix cycles go by that); the exact variants skip every test of a
// column against head_dim and load 16 bytes where the others load 4.
template <int DH, typename F>
static hipError_t by_mode(int D, int load, F&& f) {
  std::integral_constant<int, DH> dh;
  if (load == kLoadScalar) return f(dh, std::integral_constant<int, kF32Far>());
  return D == DH ? f(dh, std::integral_constant<int, kF32Exact>()) : f(dh, std::integral_constant<int, kF32Padded>());
}
template <typename F>
static hipError_t by_head_dim(int D, int load, F&& f) {
  switch ((D + 31) / 32) {
    case 1: return by_mode<32>(D, load, f);
    case 2: return by_mode<64>(D, load, f);
    case 3: return by_mode<96>(D, load, f);
    default: return by_mode<128>(D, load, f);
  }
}

hipError_t launch_fwd_f32(const FwdParams& p, int max_tiles, hipStream_t stream) {
  return by_head_dim(p.head_dim, p.load, [&](auto dh, auto mode) {
    hipLaunchKernelGGL((fwd_f32_kernel<decltype(dh)::value, decltype(mode)::value>), dim3((unsigned)(xcd_sub_grid(max_tiles * p.num_heads, kF32Split) + p.sched.service)),
                       dim3(kThreads), 0, stream, p);
    return hipGetLastError();
  });
}

hipError_t launch_bwd_f32(const BwdParams& p, int max_q_tiles, int max_k_tiles, hipStream_t stream) {
  int dev = 0, cus = 0;
  const hipError_t e = device_cus(&dev, &cus);
  if (e != hipSuccess) return e;
  return by_head_dim(p.head_dim, p.load, [&](auto dh, auto mode) {
    constexpr int DH = decltype(dh)::value;
    constexpr int kMode = decltype(mode)::value;
    constexpr size_t lds_bytes = DkvF32Lds<DH>::kFloats * sizeof(float);
    static std::atomic<uint64_t> lds_done{0};
    const hipError_t r = raise_lds_limit(&bwd_dkv_f32_kernel<DH, kMode>, lds_done, dev, lds_bytes);
    if (r != hipSuccess) return r;
    hipLaunchKernelGGL((bwd_dq_f32_kernel<DH, kMode>), dim3((unsigned)xcd_sub_grid(max_q_tiles * p.num_heads, kF32Split)), dim3(kThreads), 0, stream, p);
    hipLaunchKernelGGL((bwd_dkv_f32_kernel<DH, kMode>), dim3((unsigned)xcd_sub_grid(max_k_tiles * p.num_heads, kF32KeySplit)), dim3(kThreads), lds_bytes, stream, p);
    return hipGetLastError();
  });
}

}  // namespace sba
