// fp32 path: the same operator for fp32 inputs, everything held and summed in fp32.
//
// Products.  An fp32 number is the sum of three bf16 numbers; of the nine products of two such triples the six that matter are formed
// on the bf16 matrix instruction (v_mfma_f32_32x32x16_bf16: exact products, fp32 sums), which takes 192 cycles for a 32 x 32 x 16 block
// where v_mfma_f32_32x32x2_f32 takes 512.  A sum of three terms or more is the more accurate one (fewer roundings; rms error of a sum of
// positive products, in 2^-24, triples and fp32 instruction: 0.58 and 0.43 for 1 term, 0.53 and 0.50 for 2, 0.50 and 0.55 for 3, 0.46 and
// 0.78 for 8, 2.3 and 2.9 for 128).  Fewer terms stay with the fp32 instruction: the first 32 rows of a sequence in the forward and in dQ, its
// keys that fewer than 32 rows behind their block see in dK/dV, and head_dims 1 and 2.  Against float64, 8 heads, 6 sequences of up to
// 500 tokens, head_dims 16 to 128, three kinds of values: rms error of o, dq, dk, dv 0.80 to 0.93 of the fp32 instruction's.  Workgroups
// that meet numbers which triples do not hold (see Split) run again on the fp32 instruction.
// What bounds it: per 32 x 32 block at head_dim 128 the forward needs 3072 matrix cycles and 1300 vector instructions (5200 cycles), 700 of
// them to split K and V, which every workgroup of 32 rows does for itself; two waves per SIMD overlap the two to about 70 %.
// Consequences for the design:
//   * no tile is shared between waves: an operand goes from global memory straight into the registers of the wave that
//     uses it, a phase ahead of its use, in the registers the phase before has consumed.  One barrier per 128 keys; two waves
//     per SIMD cover each other's element-wise math.
//   * the unit of work is small (32 query rows, or 32 keys, per workgroup of four waves), because the longest row
//     would otherwise be the critical path: 32 rows of 2048 keys are 64 blocks, one wave 0.1 ms.
//     The four waves split the KEYS of the forward and
//     of dQ (sub-tiles of 32 dealt round robin, one scalar per row exchanged per step) and the ROWS of dK/dV (nothing
//     exchanged), and add their partial results through LDS at the end, in a fixed order: bit-reproducible.
// Measured: 12 heads x 128, 6143 tokens in sequences of up to 2048, forward + backward: 1.01 ms with the fp32 instruction, 0.85 ms
// with triples (forward 0.20, dQ 0.28, dK/dV 0.36); head_dim 64 0.53 and 0.45, 96 0.75 and 0.63, 127 1.20 and 0.95, 32 (4 heads) 0.175 and
// 0.151.  All nine products but l x l, with the small ones in a sum of their own, would halve the errors and cost more than the gain: 1.09 ms.
//
//   fwd_f32_kernel     : keys swept in reverse from the diagonal (as sb_varlen_fwd.py:155-165), running product per row;
//                        records the product above every 32-key sub-tile in `carry`.
//   bwd_dq_f32_kernel  : keys swept forwards; A from the recorded products, g = A (dO.v - drem), C = prefix sum of g,
//                        dz = g - sigma C (sb_varlen_bwd.py:438-447), dQ += dZ K; records C below every sub-tile.
//   bwd_dkv_f32_kernel : key-stationary; dV += P^T dO, dK += dZ^T Q over the rows that see the keys.
//
// Register layout: S^T = K Q^T as in the 16-bit kernels (lane l owns query l%32 and the 16 consecutive keys
// 16*(l/32) + r).  The contraction index of an MFMA is split between the half-waves, and which element it
// stands for is free as long as both operands agree.
//   fp32 instruction, k = l/32: over head_dim d = 8*i + 4*(l/32) + t for MFMA 4*i + t, so a lane reads 16-byte pieces of its row from
//     LDS; over keys/rows index 16*(l/32) + r for MFMA r: the score registers are the A operand as they stand.
//   bf16 instruction, k = 8*(l/32) + t: over head_dim 16 consecutive columns, planes of bf16 in LDS; over keys/rows index
//     16*(l/32) + 8*i + t for MFMA i: score registers and columns of x are operands as they stand, split pair by pair.
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

enum : int { kF32Padded = 0, kF32Exact = 1, kF32Far = 2, kF32Quads = 3 };      // how rows are read, see Operand

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int r = 0; r < 16; r++) z[r] = 0.f;
  return z;
}
// The lane's number, computed where it is used: the addresses that follow from it would cost registers that the loops do not have.
__device__ __forceinline__ int this_lane() {
  int r;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(r));
  return r;
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
// kF32Exact: head_dim == DH.  kF32Quads: a multiple of 4.  kF32Padded: any; an element beyond head_dim is asked for outside the buffer
// and reads as zero.
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
// Returns whether this thread stored a sum that calls for the other engine (see Split).
template <class E, int DH, int kMode>
__device__ __forceinline__ bool reduce_store_f32(float* lds, const f32x16 (&acc)[DH / 32], float scale, float* out, int64_t stride,
                                                 int rows, int D, const float* add = nullptr, int64_t add_stride = 0,
                                                 const float* add_scale = nullptr) {
  constexpr int NB = DH / 32, kStride = DH + 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, half = lane >> 5, col = lane & 31;
  bool odd = false;
  __syncthreads();
  float* mine = lds + wave * 32 * kStride;
#pragma unroll
  for (int r = 0; r < 16; r++)
#pragma unroll
    for (int dt = 0; dt < NB; dt++)
      mine[(8 * (r >> 2) + 4 * half + (r & 3)) * kStride + E::out_col(dt, col)] = acc[dt][r];
  __syncthreads();
  for (int idx = threadIdx.x; idx < 32 * (DH / 4); idx += kThreads) {
    const int row = idx / (DH / 4), d0 = (idx % (DH / 4)) * 4;
    if (row >= rows || d0 >= D) continue;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kWaves; w++) v += *reinterpret_cast<const f32x4*>(lds + (w * 32 + row) * kStride + d0);
#pragma unroll
    for (int t = 0; t < 4; t++) {
      if (kMode == kF32Exact || d0 + t < D) odd |= E::odd_sum(v[t]);
      v[t] *= E::kDown * E::kDown;
    }
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
  return odd;
}

// The two ways to form the products.  x: the registers of the streamed operand.
//   stage    : 32 rows into LDS as the resident operand of score() (kRows: as its A operand, whose row m is key mfma_row_to_key32(m))
//   score    : (rows in x) . (resident rows), contracted over head_dim (kGrad: dP, times 1 / kDown); x then holds `next`
//   contract : acc[dt] += a . x, contracted over 32 rows, a times 1 / kDown, the result times 1 / kDown^2; x then holds `next` if `more`
template <int DH, int kMode>
struct Plain {
  typedef Operand<DH, kMode> Op;
  typedef float Stream[DH / 2];
  static constexpr bool kSplit = false, kLaid = false;
  static constexpr float kUp = 1.f, kDown = 1.f;
  static __device__ __forceinline__ bool odd_sum(float) { return false; }
  static constexpr int kResident = 32 * (DH + 4), kTurn = Parts<DH>::kTurn;      // floats
  static __device__ __forceinline__ int out_col(int dt, int col) { return sba::out_col<DH>(dt, col); }
  static __device__ __forceinline__ Op op(const float* base, int64_t stride, int first, int rows_total, int half, int col, int D) {
    return operand<DH, kMode>(base, stride, first, rows_total, half, col, D);
  }
  template <bool kScore>
  static __device__ __forceinline__ void fill(float (&x)[DH / 2], const Op& o) { o.fill(x); }
  template <bool kRows>
  static __device__ __forceinline__ bool stage(float* lds, const Rows32& s, int D) {
    stage_rows<DH, kMode>(lds, s, D);
    return false;
  }
  template <bool kLdsIsA, bool kNextScore, bool kGrad>
  static __device__ __forceinline__ f32x16 score(float (&x)[DH / 2], float* turn, const float* resident, int half, int col, const Op& next,
                                                 const Op& late, bool has_late, uint64_t& odd) {
    const int key = mfma_row_to_key32(col);
    return score_phase<DH, kMode, kLdsIsA>(x, turn, kLdsIsA ? col : key, resident + (kLdsIsA ? key : col) * (DH + 4), half, col, next, late, has_late);
  }
  template <bool kNextScore>
  static __device__ __forceinline__ void contract(f32x16 (&acc)[DH / 32], const float (&a)[16], float (&x)[DH / 2], const Op& next, bool more,
                                                  const Op& late, bool has_late) {
    contract_phase<DH, kMode>(acc, a, x, next, more, late, has_late);
  }
};

// An fp32 number as the sum of three bf16 numbers, each the one before's rounding error rounded: 26 bits.  (Numbers whose first part
// rounds to infinity have none; what comes of them is not a number.)  Pairs of numbers; the residuals are exact.
struct Split3 { uint32_t h, m, l; };
__device__ __forceinline__ Split3 split3(float x0, float x1) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  auto round = [](float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2)); };
  auto low = [](uint32_t v) { return __builtin_bit_cast(float, v << 16); };
  auto high = [](uint32_t v) { return __builtin_bit_cast(float, v & 0xffff0000u); };
  Split3 r;
  r.h = round(x0, x1);
  const float m0 = x0 - low(r.h), m1 = x1 - high(r.h);
  r.m = round(m0, m1);
  r.l = round(m0 - low(r.m), m1 - high(r.m));
  return r;
}

// Products of triples.  What they do not hold: numbers beyond the largest bf16 number (and infinities), whose triples are not numbers,
// and the last bits of numbers below 2^-102, whose last parts would be no normal numbers.
//   Resident rows (Q, dO; K, V): a workgroup calls for the fp32 instruction (`odd`) if an element is outside 2^-80 .. 2^80.
//   Streamed rows: the operand of dP and those of the contractions are scaled by 2^24 before they are split (kUp), and so are the weights
//     and their gradients they are contracted with: no fp32 number loses a bit.  dP and the results are scaled back.  What is too large
//     for that makes infinities or no numbers, in results that rows or keys of the workgroup store: they call for the fp32 instruction.
//   The operand of the logits is not scaled: a part lost there is below 2^-126, times 2^80 of the resident row and 128 columns 2^-39,
//     times the logit scale (at most 2^10 here, see fp32_products_only) nothing that a logit's effect could show.  Logits that are no
//     numbers call for the fp32 instruction, infinite ones saturate as they do there.
// Cost of the scaling: 12 heads x 128, 6143 tokens, forward 230 -> 230 us, dQ 315 -> 323, dK/dV 402 -> 408.
// The residuals are taken with shifts and subtractions: v_dot2_f32_bf16 does it in one instruction instead of two, but not beside
// MFMAs (12 heads, 6143 tokens: 828 us against 800).
template <int DH, int kMode>
struct Split {
  typedef typename Elem<__bf16>::vec8 vec8;
  typedef float Stream[DH / 2];
  static constexpr bool kSplit = true, kLaid = false;
  static constexpr float kUp = 0x1p24f, kDown = 0x1p-24f;
  static __device__ __forceinline__ bool odd(float x) { return x != 0.f && !(fabsf(x) >= 0x1p-80f && fabsf(x) <= 0x1p80f); }
  static __device__ __forceinline__ bool odd_sum(float x) { return !(fabsf(x) < INFINITY); }
  static constexpr int NB = DH / 32, kPlane = 2048, kPanel = 3 * kPlane;      // bytes; a panel: 3 planes of [32 rows][32 columns]
  static constexpr int kResident = NB * kPanel / 4, kTurn = kPanel / 4;       // floats
  static __device__ __forceinline__ int out_col(int dt, int col) { return NB * col + dt; }

  // 32 rows in DH/2 registers per lane.  For score(): piece (p, i) is rows 8 i + lane/8, columns 32 p + 4 (lane%8) .. +3, in registers
  // 16 p + 4 i.  For contract(): piece r is row 16 half + r, columns NB (lane%32) .. +NB-1, in registers NB r.
  struct Op {
    Rows32 src;
    uint32_t voff_s, voff_c;
    int lane, D;
    // kN numbers from byte voff on, which are columns d to d + kN - 1; zero if all are beyond head_dim.  A piece that head_dim cuts holds
    // what lies behind the row (within the rows' memory, or zero beyond the resource's end), or, kZero, zeros there.
    template <int kN, bool kZero>
    __device__ __forceinline__ void load(float* y, uint32_t voff, uint32_t soff, int d) const {
      const uint32_t vo = kMode == kF32Exact || d < D ? voff : (uint32_t)kOutside;
      if constexpr (kN == 1) {
        y[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(src.rsrc, vo, soff, 0));
      } else {
        typedef __attribute__((ext_vector_type(kN))) float vec;
        vec v;
        if constexpr (kN == 2) v = __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b64(src.rsrc, vo, soff, 0));
        else if constexpr (kN == 3) v = __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b96(src.rsrc, vo, soff, 0));
        else v = __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b128(src.rsrc, vo, soff, 0));
#pragma unroll
        for (int c = 0; c < kN; c++) y[c] = !kZero || kMode != kF32Padded || c == 0 || d + c < D ? v[c] : 0.f;
      }
    }
    __device__ __forceinline__ void score_piece(float (&x)[DH / 2], int p, int i) const {
      load<4, true>(x + 16 * p + 4 * i, voff_s + 128 * p, 8u * (uint32_t)i * src.stride_bytes, 32 * p + 4 * (lane & 7));
    }
    __device__ __forceinline__ void contract_piece(float (&x)[DH / 2], int r) const {
      load<NB, false>(x + NB * r, voff_c, (uint32_t)r * src.stride_bytes, NB * (lane & 31));
    }
    // The pieces whose registers are free once those below `to` are, and were not once those below `from` were.
    template <bool kScore>
    __device__ __forceinline__ void refill(float (&x)[DH / 2], int from, int to) const {
      if (kScore) {
#pragma unroll
        for (int j = 0; j < DH / 8; j++)
          if (4 * j + 4 > from && 4 * j + 4 <= to) score_piece(x, j >> 2, j & 3);
      } else {
#pragma unroll
        for (int r = 0; r < 16; r++)
          if (NB * r + NB > from && NB * r + NB <= to) contract_piece(x, r);
      }
    }
  };
  static __device__ __forceinline__ Op op(const float* base, int64_t stride, int first, int rows_total, int half, int col, int D) {
    const Rows32 s = rows32(base, stride, first, rows_total, D);
    const int lane = this_lane();
    return Op{s, (uint32_t)(lane >> 3) * s.stride_bytes + 16u * (lane & 7), 16u * (uint32_t)(lane >> 5) * s.stride_bytes + 4u * NB * (lane & 31), lane, D};
  }
  template <bool kScore>
  static __device__ __forceinline__ void fill(float (&x)[DH / 2], const Op& o) { o.template refill<kScore>(x, 0, DH / 2); }

  // Panels: 64-byte rows whose 16-byte chunks are XORed with (row >> 2) & 3: no bank is met twice by row reads.
  static __device__ __forceinline__ void put(unsigned char* at, float a, float b, float c, float d, float up = 1.f) {
    const Split3 u = split3(up * a, up * b), v = split3(up * c, up * d);
    *reinterpret_cast<u32x2*>(at) = u32x2{u.h, v.h};
    *reinterpret_cast<u32x2*>(at + kPlane) = u32x2{u.m, v.m};
    *reinterpret_cast<u32x2*>(at + 2 * kPlane) = u32x2{u.l, v.l};
  }
  template <bool kRows>
  static __device__ __forceinline__ bool stage(float* lds, const Rows32& s, int D) {
    bool any = false;
    unsigned char* const at = (unsigned char*)lds;
    for (int idx = threadIdx.x; idx < 32 * (DH / 4); idx += kThreads) {
      const int row = idx / (DH / 4), d = (idx % (DH / 4)) * 4;
      const Op o{s, 0, 0, 0, D};
      float v[4];
      o.template load<4, true>(v, (uint32_t)row * s.stride_bytes + 4 * d, 0, d);
      const int m = kRows ? 8 * ((row & 15) >> 2) + 4 * (row >> 4) + (row & 3) : row;
      put(at + (d >> 5) * kPanel + m * 64 + ((((d >> 3) & 3) ^ ((m >> 2) & 3)) << 4) + 2 * (d & 4), v[0], v[1], v[2], v[3]);
#pragma unroll
      for (int c = 0; c < 4; c++) any |= odd(v[c]);
    }
    return any;
  }
  // A wave's 32 x 32 piece p of 32 rows, in x as score_piece() loads it, into a panel of its own: rows 8 i + lane/8 go to their own place,
  // or (as the A operand) to that of their key.
  template <bool kLdsIsA>
  static __device__ __forceinline__ int turn_place(int lane) {
    const int l8 = lane >> 3, chunk = (lane & 7) >> 1, sub = 8 * (lane & 1);
    return kLdsIsA ? l8 * 64 + ((chunk ^ (l8 >> 2)) << 4) + sub : (8 * (l8 >> 2) + (l8 & 3)) * 64 + ((chunk ^ (2 * (l8 >> 2))) << 4) + sub;
  }
  template <bool kLdsIsA>
  static __device__ __forceinline__ void put_panel(unsigned char* mine, int w0, const float (&x)[DH / 2], int p, float up) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int w = kLdsIsA ? (w0 ^ (32 * (i & 1))) + 512 * i : (w0 ^ (16 * (i >> 1))) + 1024 * (i & 1) + 256 * (i >> 1);
      const float* y = x + 16 * p + 4 * i;
      put(mine + w, y[0], y[1], y[2], y[3], up);
    }
  }
  // Where this lane's part of an operand over 16 columns starts in a panel (the other 16 columns: ^ 32).
  static __device__ __forceinline__ int row_place(int lane) { return (lane & 31) * 64 + (((lane >> 5) ^ ((lane >> 2) & 3)) << 4); }
  // 8 numbers as the three planes of an operand.
  template <typename At>
  static __device__ __forceinline__ void planes(At&& at, vec8 (&out)[3]) {
    u32x4 v[3];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const Split3 u = split3(at(2 * t), at(2 * t + 1));
      v[0][t] = u.h; v[1][t] = u.m; v[2][t] = u.l;
    }
#pragma unroll
    for (int j = 0; j < 3; j++) out[j] = as_vec8<__bf16>(v[j]);
  }
  // The six products that matter, the small ones first.  (m x l twice and l x l are left out, 2^-25 of the product at most.)
  static __device__ __forceinline__ f32x16 six(const vec8 (&a)[3], const vec8 (&b)[3], f32x16 c) {
    c = Elem<__bf16>::mfma(a[2], b[0], c);
    c = Elem<__bf16>::mfma(a[0], b[2], c);
    c = Elem<__bf16>::mfma(a[1], b[1], c);
    c = Elem<__bf16>::mfma(a[1], b[0], c);
    c = Elem<__bf16>::mfma(a[0], b[1], c);
    return Elem<__bf16>::mfma(a[0], b[0], c);
  }
  template <bool kLdsIsA, bool kNextScore, bool kGrad>
  static __device__ __forceinline__ f32x16 score(float (&x)[DH / 2], float* turn, const float* resident, int half, int col, const Op& next,
                                                 const Op&, bool, uint64_t& odd) {
    f32x16 acc = zero16();
    unsigned char* const mine = (unsigned char*)turn;
    const unsigned char* const res = (const unsigned char*)resident;
    const int lane = this_lane(), w0 = turn_place<kLdsIsA>(lane), row_a = row_place(lane);
#pragma unroll
    for (int p = 0; p < NB; p++) {
      put_panel<kLdsIsA>(mine, w0, x, p, kGrad ? kUp : 1.f);
      next.template refill<kNextScore>(x, 16 * p, 16 * p + 16);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < 2; kk++) {
        vec8 a[3], b[3];
#pragma unroll
        for (int j = 0; j < 3; j++) {
          const int at = kk ? row_a ^ 32 : row_a;
          const vec8 u = *reinterpret_cast<const vec8*>(mine + j * kPlane + at), v = *reinterpret_cast<const vec8*>(res + p * kPanel + j * kPlane + at);
          a[j] = kLdsIsA ? v : u;
          b[j] = kLdsIsA ? u : v;
        }
        acc = six(a, b, acc);
      }
    }
    if (!kGrad) {      // (dP that is not a number makes results that are none)
#pragma unroll
      for (int r = 0; r < 16; r += 2) odd |= __ballot(__builtin_isunordered(acc[r], acc[r + 1]));
    }
    return acc;
  }
  template <bool kNextScore>
  static __device__ __forceinline__ void contract(f32x16 (&acc)[DH / 32], const float (&a)[16], float (&x)[DH / 2], const Op& next, bool more,
                                                  const Op&, bool) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      vec8 av[3];
      planes([&](int t) { return a[8 * i + t]; }, av);
#pragma unroll
      for (int dt = 0; dt < NB; dt++) {
        vec8 bv[3];
        planes([&](int t) { return kUp * x[(8 * i + t) * NB + dt]; }, bv);
        acc[dt] = six(av, bv, acc[dt]);
      }
      next.template refill<kNextScore>(x, 8 * NB * i, 8 * NB * (i + 1));
      __builtin_amdgcn_sched_barrier(0);
    }
  }
};

// Products of triples whose streamed operand a kernel in front has split and laid out as the matrix instruction takes it (lay_f32_kernel): a
// wave loads what it needs straight into operand registers, three planes of 1 KB per six products, kAhead operands ahead of their use.  The numbers
// and the order of the sums are Split's, and so are the bits.
// What it saves: a workgroup of 32 rows or keys splits every operand that streams past it for itself, which in dQ is 1180 of 1900 vector-ALU
// instructions per 32 x 32 block (4608 matrix cycles) and in dK/dV 1540 of 2800 (6144), and turns those of the scores round through LDS.  What it costs: six
// bytes per element from the L2 instead of four, and the planes (the line between the two stands with laid_pieces in sba_api.hip).  Long sequences
// alone on the chip run at the rate of their instructions (one head x 8192 x 128: 10 us of a wave's 32 x 32 blocks in dQ and dK/dV together); many, where
// a quarter of the reads miss the L2, wait for those: 12 heads x 128, 6143 tokens, dQ 297 -> 237 us, dK/dV 380 -> 290, laying out 45 + 65.  Two
// operands ahead instead of four 260 and 319; the resident operand read from LDS one ahead 236 and 305; one workgroup per compute unit
// 423 (dK/dV); raised wave priority in either phase no change.
// Training passes, us: one head x 8192 x 128 1303 -> 939, 2 x 4096 x 50 445 -> 368, 8 x 4096 x 128 1160 -> 981, 32 heads x 16384 tokens of 2048 x 128
// 9187 -> 8729.
template <int DH, int kMode>
struct Laid : Split<DH, kMode> {
  typedef Split<DH, kMode> S;
  typedef typename S::vec8 vec8;
  static constexpr bool kLaid = true;
  static constexpr int NB = S::NB, kTurn = 0;
  static constexpr int kOps = 2 * NB, kAhead = NB == 4 ? 4 : kOps < 6 ? kOps : 3;      // operands of a phase; a divisor of it
  static constexpr int kOpBytes = 3 * 1024, kTile = kOps * kOpBytes;                   // of 32 rows
  struct Op {
    __amdgpu_buffer_rsrc_t score, contract;      // from the sequence's first 32 rows on
    int at;                                      // byte of these 32 rows
  };
  struct Stream {
    u32x4 ring[kAhead][3];
    __amdgpu_buffer_rsrc_t rsrc;                 // of the phase under way
    int at;
    __device__ __forceinline__ void load(const __amdgpu_buffer_rsrc_t& r, int byte, int i) {
      const int voff = this_lane() * 16;
#pragma unroll
      for (int j = 0; j < 3; j++) ring[i % kAhead][j] = __builtin_amdgcn_raw_buffer_load_b128(r, voff + 1024 * j, byte + i * kOpBytes, 0);
    }
    __device__ __forceinline__ void take(int i, vec8 (&v)[3]) const {
#pragma unroll
      for (int j = 0; j < 3; j++) v[j] = as_vec8<__bf16>(ring[i % kAhead][j]);
    }
  };
  template <bool kScore>
  static __device__ __forceinline__ void fill(Stream& x, const Op& o) {
    x.rsrc = kScore ? o.score : o.contract;
    x.at = o.at;
#pragma unroll
    for (int i = 0; i < kAhead; i++) x.load(x.rsrc, x.at, i);
  }
  // Operand i has been used: the one kAhead further on, of this phase or the next.
  template <bool kNextScore>
  static __device__ __forceinline__ void step(Stream& x, const Op& next, int i, bool more = true) {
    if (i + kAhead < kOps) x.load(x.rsrc, x.at, i + kAhead);
    else if (more) x.load(kNextScore ? next.score : next.contract, next.at, i + kAhead - kOps);
    if (i + 1 == kOps) {
      x.rsrc = kNextScore ? next.score : next.contract;
      x.at = next.at;
    }
  }
  template <bool kLdsIsA, bool kNextScore, bool kGrad>
  static __device__ __forceinline__ f32x16 score(Stream& x, float*, const float* resident, int, int, const Op& next, const Op&, bool, uint64_t& odd) {
    f32x16 acc = zero16();
    const unsigned char* const res = (const unsigned char*)resident;
    const int row_a = S::row_place(this_lane());
#pragma unroll
    for (int i = 0; i < kOps; i++) {
      vec8 u[3], v[3];
      x.take(i, u);
#pragma unroll
      for (int j = 0; j < 3; j++) v[j] = *reinterpret_cast<const vec8*>(res + (i >> 1) * S::kPanel + j * S::kPlane + (i & 1 ? row_a ^ 32 : row_a));
      acc = kLdsIsA ? S::six(v, u, acc) : S::six(u, v, acc);
      step<kNextScore>(x, next, i);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!kGrad) {
#pragma unroll
      for (int r = 0; r < 16; r += 2) odd |= __ballot(__builtin_isunordered(acc[r], acc[r + 1]));
    }
    return acc;
  }
  template <bool kNextScore>
  static __device__ __forceinline__ void contract(f32x16 (&acc)[NB], const float (&a)[16], Stream& x, const Op& next, bool more, const Op&, bool) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      vec8 av[3];
      S::planes([&](int t) { return a[8 * i + t]; }, av);
#pragma unroll
      for (int dt = 0; dt < NB; dt++) {
        vec8 bv[3];
        x.take(i * NB + dt, bv);
        acc[dt] = S::six(av, bv, acc[dt]);
        step<kNextScore>(x, next, i * NB + dt, more);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
};
// The 32-row pieces of a head's sequences in such a plane: sequences one after the other, each from a piece of its own on (packed: what starts at
// token t of the batch as its s-th sequence at piece t / 32 + s, which is beyond the last piece of the one before).
__device__ __forceinline__ int64_t laid_piece(const LaidPlanes& l, const Tile& tile) {
  return l.per_seq ? (int64_t)tile.seq_id * l.per_seq : (int64_t)(tile.seq_start >> 5) + tile.seq_id;
}
template <int DH, int kMode>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t laid_rows(const LaidPlanes& l, const Tile& tile, int head, int plane) {
  constexpr int kTile = Laid<DH, kMode>::kTile;
  const int64_t first = laid_piece(l, tile), left = min(l.pieces - first, (int64_t)(0x7fffffff / kTile));
  return __builtin_amdgcn_make_buffer_rsrc(l.base + (plane * l.plane_pieces + head * l.pieces + first) * kTile, 0, (int)left * kTile, 0x00020000);
}

// Bound by memory: it reads 512 and writes up to 3 KB per row at head_dim 128 (12 heads, 6143 tokens: k and v 45 us, q and d_o 65, 4.6 TB/s).
// 32 rows of q and d_o (kKeys: k and v) as operands: an MFMA operand is 64 lanes x 16 bytes, its three planes follow each other.  Planes: 0 and
// 1 q (k) over its columns and over its rows, 2 d_o (v) over its columns, 3 d_o over its rows.  A wave per 32 rows and tensor.
template <int DH, int kMode, bool kKeys>
__global__ __launch_bounds__(kThreads, 2) void lay_f32_kernel(BwdParams p) {
  typedef Split<DH, kMode> S;
  typedef Laid<DH, kMode> Out;
  __shared__ __attribute__((aligned(16))) unsigned char lds[kWaves * S::kPanel];
  int head, slot, second;
  xcd_head_tile_sub(blockIdx.x, 2, p.num_heads, &head, &slot, &second);
  if (slot >= p.counts[kCountQ]) return;
  const Tile tile = p.q_tiles[slot];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, col = lane & 31;
  const int row0 = tile.origin + 32 * wave;
  if (row0 >= tile.seq_len) return;
  const TensorRef& t = kKeys ? (second ? p.v : p.k) : (second ? p.d_o : p.q);
  const float* base = (const float*)t.ptr + tile.seq_id * t.sb + head * t.sh + (int64_t)tile.seq_start * t.st;
  const typename S::Op o = S::op(base, t.st, row0, tile.seq_len, half, col, p.head_dim);
  unsigned char* const mine = lds + wave * S::kPanel;
  const int piece = (row0 >> 5) * Out::kTile;
  auto put = [&](const __amdgpu_buffer_rsrc_t& out, int op, int j, u32x4 v) {
    __builtin_amdgcn_raw_buffer_store_b128(v, out, lane * 16 + piece + op * Out::kOpBytes + 1024 * j, 0, 0);
  };
  float x[DH / 2];
  S::template fill<true>(x, o);
  {
    const __amdgpu_buffer_rsrc_t out = laid_rows<DH, kMode>(p.laid, tile, head, second ? 2 : 0);
    const int w0 = S::template turn_place<!kKeys>(lane), row_a = S::row_place(lane);
#pragma unroll
    for (int c = 0; c < S::NB; c++) {
      S::template put_panel<!kKeys>(mine, w0, x, c, second ? S::kUp : 1.f);
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int kk = 0; kk < 2; kk++)
#pragma unroll
        for (int j = 0; j < 3; j++) put(out, 2 * c + kk, j, *reinterpret_cast<const u32x4*>(mine + j * S::kPlane + (kk ? row_a ^ 32 : row_a)));
      __builtin_amdgcn_wave_barrier();
    }
  }
  if (kKeys && second) return;
  S::template fill<false>(x, o);
  const __amdgpu_buffer_rsrc_t out = laid_rows<DH, kMode>(p.laid, tile, head, second ? 3 : 1);
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int dt = 0; dt < S::NB; dt++) {
      typename S::vec8 v[3];
      S::planes([&](int t) { return S::kUp * x[(8 * i + t) * S::NB + dt]; }, v);
#pragma unroll
      for (int j = 0; j < 3; j++) put(out, i * S::NB + dt, j, __builtin_bit_cast(u32x4, v[j]));
    }
}

template <int DH, int kMode, bool kLaid = false>
using Engine = typename std::conditional<kMode == kF32Far, Plain<DH, kMode>, typename std::conditional<kLaid, Laid<DH, kMode>, Split<DH, kMode>>::type>::type;

// LDS of the row-stationary kernels: kTiles tiles of 32 rows and the waves' scratch; the final sums lie over both.
constexpr int most(int a, int b) { return a > b ? a : b; }
template <class E, int DH, int kTiles>
struct RowsF32Lds {
  static constexpr int kFloats = most(kTiles * E::kResident + kWaves * E::kTurn, kWaves * 32 * (DH + 4));
};
template <int DH, int kMode, int kTiles>
constexpr int kRowsF32 = most(RowsF32Lds<Plain<DH, kMode>, DH, kTiles>::kFloats, RowsF32Lds<Engine<DH, kMode>, DH, kTiles>::kFloats);

// Where the products were split: whether any wave met what the fp32 matrix instruction treats otherwise (the workgroup agrees).
__device__ __forceinline__ bool any_odd(uint64_t odd, bool mine) { return __syncthreads_or((int)(odd != 0) | (int)mine) != 0; }

template <class E, int DH, int kMode>
__device__ __forceinline__ bool fwd_f32_rows(const FwdParams& p, const Tile& tile, int head, int q0, float* lds, float (&xch)[2][kWaves][32], float (&rem_lds)[32]) {
  constexpr int NB = DH / 32;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, col = lane & 31;
  const int L = tile.seq_len, ac = p.attend_current, D = p.head_dim;
  const int64_t tok0 = tile.seq_start;
  const float* qb = (const float*)p.q.ptr + tile.seq_id * p.q.sb + head * p.q.sh + tok0 * p.q.st;
  const float* kb = (const float*)p.k.ptr + tile.seq_id * p.k.sb + head * p.k.sh + tok0 * p.k.st;
  const float* vb = (const float*)p.v.ptr + tile.seq_id * p.v.sb + head * p.v.sh + tok0 * p.v.st;
  const int64_t n_qt = (L + kBlockQ - 1) / kBlockQ;
  float* carry = p.carry ? p.carry + (int64_t)head * p.carry_head_stride + tile.carry_base : nullptr;

  const int qi = q0 + col;
  const int last_key = min(q0 + kF32Rows, L) - 2 + ac;
  const int n_sub = last_key < 0 ? 0 : last_key / 32 + 1, n_steps = (n_sub + kWaves - 1) / kWaves;
  auto k_of = [&](int u) { return E::op(kb, p.k.st, 32 * u, L, half, col, D); };
  auto v_of = [&](int u) { return E::op(vb, p.v.st, 32 * u, L, half, col, D); };
  typename E::Stream x;
  // Wave w takes sub-tile n_sub - 1 - (4 t + w) in step t.
  int U = n_sub - 1 - wave;
  if (U >= 0) E::template fill<true>(x, k_of(U));
  bool staged = E::template stage<false>(lds, rows32(qb, p.q.st, q0, L, D), D);
  float* turn = lds + E::kResident + wave * E::kTurn;
  f32x16 oacc[NB];
#pragma unroll
  for (int dt = 0; dt < NB; dt++) oacc[dt] = zero16();
  uint64_t odd = 0;
  float prod = 1.f;      // product over the keys of the steps done so far
  __syncthreads();
  for (int t = 0; t < n_steps; ++t, U -= kWaves) {
    const int me = this_lane(), half = me >> 5, col = me & 31, qi = q0 + col;
    float beta[16], pe[16];
    float run = 1.f, oth = 1.f;
    if (U >= 0) {
      const f32x16 s = E::template score<false, false, false>(x, turn, lds, half, col, v_of(U), k_of(U), t > 0, odd);
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
      const float seed = E::kUp * (half ? above : above * oth);      // the upper half-wave holds the higher keys
#pragma unroll
      for (int r = 0; r < 16; r++) pe[r] = beta[r] * (pe[r] * seed);
      E::template contract<true>(oacc, pe, x, k_of(U >= kWaves ? U - kWaves : n_sub), U >= kWaves, k_of(U), false);
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
  const bool stored = reduce_store_f32<E, DH, kMode>(lds, oacc, 1.f, ob, p.o.st, L - q0, D, p.add_rem ? vb + (int64_t)q0 * p.v.st : nullptr, p.v.st, rem_lds);
  return E::kSplit && any_odd(odd, stored | staged);
}

// (Width 96 keeps three waves per SIMD by spilling up to 29 registers: forward, 12 heads x 80 148 us, with two waves 167; x 96 165 and 167;
// padded pieces, x 95 165 and 172, but 4 heads 85 and 77.)
template <int DH, int kMode>
__global__ __launch_bounds__(kThreads, DH == 96 ? 3 : 2) void fwd_f32_kernel(FwdParams p) {
  __shared__ __attribute__((aligned(16))) float lds[kRowsF32<DH, kMode, 1>];      // Q rows and the waves' scratch, then the final sums
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
  const int q0 = tile.origin + sub * kF32Rows;
  if (q0 >= tile.seq_len) return;
  if (p.fp32_products || q0 == 0 || fwd_f32_rows<Engine<DH, kMode>, DH, kMode>(p, tile, head, q0, lds, xch, rem_lds)) fwd_f32_rows<Plain<DH, kMode>, DH, kMode>(p, tile, head, q0, lds, xch, rem_lds);
}

// What streams past a workgroup of the backward: the operand of 32 rows from 32 u on, as E takes it.
template <class E, int DH, int kMode>
__device__ __forceinline__ auto streamed(const LaidPlanes& laid, const Tile& tile, int head, int score, int contract, const float* base, int64_t stride,
                                         int half, int col, int D) {
  if constexpr (E::kLaid) {
    const __amdgpu_buffer_rsrc_t s = laid_rows<DH, kMode>(laid, tile, head, score), c = laid_rows<DH, kMode>(laid, tile, head, contract);
    return [=](int u) { return typename E::Op{s, c, u * E::kTile}; };
  } else {
    const int L = tile.seq_len;
    return [=](int u) { return E::op(base, stride, 32 * u, L, half, col, D); };
  }
}

template <class E, int DH, int kMode>
__device__ __forceinline__ bool bwd_dq_f32_rows(const BwdParams& p, const Tile& tile, int head, int q0, float* lds, float (&xch)[2][kWaves][32]) {
  constexpr int NB = DH / 32;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, col = lane & 31;
  const int L = tile.seq_len, ac = p.attend_current, D = p.head_dim;
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
  const auto k_of = streamed<E, DH, kMode>(p.laid, tile, head, 0, 1, kb, p.k.st, half, col, D);
  const auto v_of = streamed<E, DH, kMode>(p.laid, tile, head, 2, 2, vb, p.v.st, half, col, D);
  typename E::Stream x;
  int U = wave;            // wave w takes sub-tile 4 t + w in step t
  if (U < n_sub) E::template fill<true>(x, k_of(U));
  bool staged = E::template stage<false>(lds, rows32(qb, p.q.st, q0, L, D), D);
  staged |= E::template stage<false>(lds + E::kResident, rows32(dob, p.d_o.st, q0, L, D), D);
  float* turn = lds + 2 * E::kResident + wave * E::kTurn;
  float drem = 0.f;
  if (qi < L && p.d_rem.ptr) drem = ((const float*)p.d_rem.ptr)[tile.seq_id * p.d_rem.sb + head * p.d_rem.sh + (tok0 + qi) * p.d_rem.st];
  __syncthreads();
  if (p.add_rem) {
    // The forward wrote o + rem * v: the gradient reaching rem is d_rem + d_o . v_i.
    const float* vi = vb + (int64_t)min(qi, L - 1) * p.v.st;
    float dot = 0.f;
    const float* doi = dob + (int64_t)min(qi, L - 1) * p.d_o.st;
    for (int d = half; d < D; d += 2) dot = fmaf(doi[d], vi[d], dot);
    drem += dot + other_half(dot, half);
  }
  if (wave == 0 && half == 0 && qi < L) p.drem_eff[tile.seq_id * p.drem_sb + head * p.stat_sh + tok0 + qi] = drem;

  f32x16 dqacc[NB];
#pragma unroll
  for (int dt = 0; dt < NB; dt++) dqacc[dt] = zero16();
  uint64_t odd = 0;
  float prefix = 0.f;      // sum of g over the keys of the steps done so far
  for (int t = 0; t < n_steps; ++t, U += kWaves) {
    const int me = this_lane(), half = me >> 5, col = me & 31, qi = q0 + col;
    float beta[16], dz[16];
    float tot = 0.f, fix = 0.f;
    const int64_t cslot = carry_offset(U, n_qt) + (qi - kBlockQ * (U >> 2));
    const bool active = U < n_sub;
    if (active) {
      const float prod_in = carry[cslot];
      const f32x16 s = E::template score<false, true, false>(x, turn, lds, half, col, v_of(U), k_of(U), t > 0, odd);
      const f32x16 dp = E::template score<false, false, true>(x, turn, lds + E::kResident, half, col, k_of(U), k_of(U), false, odd);
      float pe[16];
      const float run = sticks_f32(s, p.scale_log2, qi < L ? qi + ac - 32 * U - 16 * half : 0, beta, pe);
      const float oth = other_half(run, half);
      const float seed = E::kUp * (half ? prod_in : prod_in * oth);
      float acc = 0.f;
#pragma unroll
      for (int R = 0; R < 16; R++) {
        const float g = beta[R] * (pe[R] * seed) * fmaf(dp[R], E::kDown, -drem);
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
      if (half == 0) prefix_out[cslot] = E::kDown * below;
      const float fixup = below + fix;
#pragma unroll
      for (int r = 0; r < 16; r++) dz[r] -= beta[r] * fixup;
      E::template contract<true>(dqacc, dz, x, k_of(U + kWaves), U + kWaves < n_sub, k_of(U), false);
    }
  }
  float* dqb = (float*)p.dq.ptr + tile.seq_id * p.dq.sb + head * p.dq.sh + (tok0 + q0) * p.dq.st;
  const bool stored = reduce_store_f32<E, DH, kMode>(lds, dqacc, p.logit_scale, dqb, p.dq.st, L - q0, D);
  return E::kSplit && any_odd(odd, stored | staged);
}

template <int DH, int kMode, bool kLaid>
__global__ __launch_bounds__(kThreads, 2) void bwd_dq_f32_kernel(BwdParams p) {
  __shared__ __attribute__((aligned(16))) float lds[kRowsF32<DH, kMode, 2>];      // Q and dO rows and the waves' scratch, then the final sums
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
  const int q0 = tile.origin + sub * kF32Rows;
  if (q0 >= tile.seq_len) return;
  if (p.fp32_products || q0 == 0 || bwd_dq_f32_rows<Engine<DH, kMode, kLaid>, DH, kMode>(p, tile, head, q0, lds, xch)) bwd_dq_f32_rows<Plain<DH, kMode>, DH, kMode>(p, tile, head, q0, lds, xch);
}

template <class E, int DH>
struct DkvF32Lds {
  static constexpr int kK = 0, kV = kK + E::kResident;                                // the workgroup's keys
  static constexpr int kTr = kV + E::kResident;                                       // per wave: operand scratch; P^T, dZ^T
  static constexpr int kTrWave = most(E::kTurn, 32 * kF32TrStride);
  static constexpr int kRem = most(kTr + kWaves * kTrWave, kWaves * 32 * (DH + 4));   // (the final sums lie over the above) rem of 32 rows
  static constexpr int kFloats = kRem + 32;
};

template <class E, int DH, int kMode>
__device__ __forceinline__ bool bwd_dkv_f32_keys(const BwdParams& p, const Tile& tile, int head, int k0, float* lds) {
  constexpr int NB = DH / 32;
  typedef DkvF32Lds<E, DH> Lds;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, col = lane & 31;
  const int L = tile.seq_len, ac = p.attend_current, D = p.head_dim;
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

  const auto q_of = streamed<E, DH, kMode>(p.laid, tile, head, 0, 1, qb, p.q.st, half, col, D);
  const auto do_of = streamed<E, DH, kMode>(p.laid, tile, head, 2, 3, dob, p.d_o.st, half, col, D);
  // Row blocks of 32 that see these keys: from the last one down to the one that holds the keys' own rows; wave w takes every
  // fourth.  (Downwards the loop needs one bound fewer in registers: 20 instead of 64 of them spilled at head_dim 128, 2 % of
  // the pass.)
  const int nb = k0 + 1 - ac < L ? (L + 31) / 32 : 0;
  int b = nb - 1 - wave;
  typename E::Stream x;
  if (b >= U) E::template fill<true>(x, q_of(b));
  // K and V of the 32 keys stay in LDS for the A operands of S^T and dP^T.
  bool staged = E::template stage<true>(lds + Lds::kK, rows32(kb, p.k.st, k0, L, D), D);
  staged |= E::template stage<true>(lds + Lds::kV, rows32(vb, p.v.st, k0, L, D), D);
  float* turn = lds + Lds::kTr + wave * Lds::kTrWave;
  float* tp = turn;                                        // P^T [key][row], then dZ^T

  uint64_t odd = 0;
  f32x16 dkacc[NB], dvacc[NB];
#pragma unroll
  for (int dt = 0; dt < NB; dt++) { dkacc[dt] = zero16(); dvacc[dt] = zero16(); }
  __syncthreads();
  for (; b >= U; b -= kWaves) {
    const int me = this_lane(), half = me >> 5, col = me & 31, qi = 32 * b + col;
    const bool row_ok = qi < L;
    const float prod_in = carry[qi], prefix_in = prefix[qi];
    const float drem = row_ok ? drem_plane[qi] : 0.f;
    const f32x16 s = E::template score<true, true, false>(x, turn, lds + Lds::kK, half, col, do_of(b), q_of(b), b < nb - kWaves, odd);
    const f32x16 dp = E::template score<true, false, true>(x, turn, lds + Lds::kV, half, col, do_of(b), do_of(b), false, odd);
    float beta[16], pe[16], dz[16];
    const float run = sticks_f32(s, p.scale_log2, row_ok ? qi + ac - k0 - 16 * half : 0, beta, pe);
    const float oth = other_half(run, half);
    const float seed = E::kUp * (half ? prod_in : prod_in * oth);
    // To [key][row] order (wave-private): the contraction over rows needs a lane per key.
    float acc = 0.f;
#pragma unroll
    for (int R = 0; R < 16; R++) {
      const float a = beta[R] * (pe[R] * seed);
      const float g = a * fmaf(dp[R], E::kDown, -drem);
      tp[(16 * half + R) * kF32TrStride + col] = a;
      acc += g;
      dz[R] = g - beta[R] * acc;
    }
    const float oth_g = other_half(acc, half);
    const float fixup = E::kUp * prefix_in + (half ? oth_g : 0.f);
#pragma unroll
    for (int R = 0; R < 16; R++) dz[R] -= beta[R] * fixup;
    float y[16];
    auto transposed = [&]() {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(tp + col * kF32TrStride + 16 * half + 4 * i);
#pragma unroll
        for (int k = 0; k < 4; k++) y[4 * i + k] = v[k];
      }
    };
    transposed();
    E::template contract<false>(dvacc, y, x, q_of(b), true, q_of(b), false);
#pragma unroll
    for (int R = 0; R < 16; R++) tp[(16 * half + R) * kF32TrStride + col] = dz[R];
    transposed();
    E::template contract<true>(dkacc, y, x, q_of(b - kWaves >= U ? b - kWaves : nb), b - kWaves >= U, q_of(b), true);
  }
  float* rem_lds = lds + Lds::kRem;
  if (p.add_rem && threadIdx.x < 32 && k0 + (int)threadIdx.x < L)      // the forward wrote o + rem * v: dv_i gains rem_i * d_o_i
    rem_lds[threadIdx.x] = exp2f(p.row_stat[tile.seq_id * p.stat_sb + head * p.stat_sh + tok0 + k0 + threadIdx.x]);
  float* dvb = (float*)p.dv.ptr + tile.seq_id * p.dv.sb + head * p.dv.sh + (tok0 + k0) * p.dv.st;
  float* dkb = (float*)p.dk.ptr + tile.seq_id * p.dk.sb + head * p.dk.sh + (tok0 + k0) * p.dk.st;
  bool stored = reduce_store_f32<E, DH, kMode>(lds, dvacc, 1.f, dvb, p.dv.st, L - k0, D, p.add_rem ? dob + (int64_t)k0 * p.d_o.st : nullptr,
                               p.d_o.st, rem_lds);
  stored |= reduce_store_f32<E, DH, kMode>(lds, dkacc, p.logit_scale, dkb, p.dk.st, L - k0, D);
  return E::kSplit && any_odd(odd, stored | staged);
}

template <int DH, int kMode, bool kLaid>
__global__ __launch_bounds__(kThreads, 2) void bwd_dkv_f32_kernel(BwdParams p) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  int head, slot, sub;
  xcd_head_tile_sub(blockIdx.x, kF32KeySplit, p.num_heads, &head, &slot, &sub);
  if (slot >= p.counts[kCountK]) return;
  const Tile tile = p.k_tiles[slot];
  const int k0 = tile.origin + sub * kF32Rows;
  if (k0 >= tile.seq_len) return;
  if (p.fp32_products || k0 + 2 * kF32Rows > tile.seq_len || bwd_dkv_f32_keys<Engine<DH, kMode, kLaid>, DH, kMode>(p, tile, head, k0, lds)) bwd_dkv_f32_keys<Plain<DH, kMode>, DH, kMode>(p, tile, head, k0, lds);
}

// head_dim is rounded up to a multiple of 32 (the matrix cycles go by that); the exact variants skip every test of a
// column against head_dim, the ones for multiples of 4 those within a piece of 4 columns (training pass, 3 heads x 80: 285 us
// instead of 430).
template <int DH, typename F>
static hipError_t by_mode(int D, int load, F&& f) {
  std::integral_constant<int, DH> dh;
  if (load == kLoadScalar) return f(dh, std::integral_constant<int, kF32Far>());
  if (D == DH) return f(dh, std::integral_constant<int, kF32Exact>());
  return D % 4 ? f(dh, std::integral_constant<int, kF32Padded>()) : f(dh, std::integral_constant<int, kF32Quads>());
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
// Whether a call has too few workgroups for split products: a step of a wave takes longer with them, and more code is fetched; they pay
// where two workgroups share a compute unit (one takes 32 rows: from 8192 rows x heads on) or, but for the narrowest, where sequences are
// long.  The first 32 rows of a sequence do not use them, which moves the line for the shortest.  Split products over fp32 products,
// the three kernels' time on 256 compute units, by rows x heads / 32:
//   equal sequences of    128           256           512           2048          6143 tokens in 5 of 600 to 2048
//   head_dim 32   to 256  1.10 .. 1.11  1.08 .. 1.09  1.08          1.05 .. 1.06  1.04
//                 from 288 1.04 (384)   0.95 .. 0.99  0.98 .. 0.99  0.89 .. 0.94  0.84 .. 0.93
//   64            to 256  1.12 .. 1.14  1.07 .. 1.09  0.99 .. 1.04  0.94 .. 0.97  0.94
//                 from 288 1.05 (384)   0.95 .. 0.98  0.92          0.85 .. 0.86  0.82 .. 0.87
//   96            to 256  1.16 .. 1.18  1.07 .. 1.12  0.99 .. 1.01  0.90 .. 0.95  0.91
//                 from 288 1.10 (384)   0.93 .. 0.94  0.87 .. 0.90  0.85 .. 0.86  0.79 .. 0.84
//   128           to 256  1.14 .. 1.17  1.07 .. 1.08  1.00 .. 1.02  0.93 .. 0.94  0.92
//                 from 288 1.02 (384)   0.91 .. 0.94  0.86 .. 0.89  0.81 .. 0.84  0.78 .. 0.84
//   (1024, 300 and 700 tokens: 0.94 .. 0.99 to 256, head_dim 32 1.06; 24 of 40 tokens: 0.96 .. 1.01 at 180.)
static bool few_workgroups(int D, int64_t rows_heads, int64_t longest) {
  return rows_heads <= 32 * (longest <= 128 ? 384 : 256) && (D <= 32 || longest < 1024);
}
// ... or sums over head_dim that are too short for them, or a logit scale at which the parts that their logits lack would count (see Split).
bool fp32_products_only(int D, int64_t rows_heads, int64_t longest, float scale_log2) {
  return few_workgroups(D, rows_heads, longest) || D <= 2 || !(fabsf(scale_log2) <= 1024.f);
}

// `rows_heads`, `longest`: of the caller's call, also where the backward takes its heads through in groups, which then give the bits of one
// pass.
hipError_t launch_fwd_f32(const FwdParams& call, int64_t rows_heads, int64_t longest, int max_tiles, hipStream_t stream) {
  FwdParams p = call;
  p.fp32_products = fp32_products_only(p.head_dim, rows_heads, longest, p.scale_log2);
  return by_head_dim(p.head_dim, p.load, [&](auto dh, auto mode) {
    hipLaunchKernelGGL((fwd_f32_kernel<decltype(dh)::value, decltype(mode)::value>), dim3((unsigned)(xcd_sub_grid(max_tiles * p.num_heads, kF32Split) + p.sched.service)),
                       dim3(kThreads), 0, stream, p);
    return hipGetLastError();
  });
}

hipError_t launch_bwd_f32(const BwdParams& call, int64_t rows_heads, int64_t longest, int max_q_tiles, int max_k_tiles, hipStream_t stream) {
  BwdParams p = call;
  p.fp32_products = fp32_products_only(p.head_dim, rows_heads, longest, p.scale_log2);
  int dev = 0, cus = 0;
  const hipError_t e = device_cus(&dev, &cus);
  if (e != hipSuccess) return e;
  return by_head_dim(p.head_dim, p.load, [&](auto dh, auto mode) {
    constexpr int DH = decltype(dh)::value;
    constexpr int kMode = decltype(mode)::value;
    constexpr size_t lds_bytes = most(DkvF32Lds<Plain<DH, kMode>, DH>::kFloats, DkvF32Lds<Engine<DH, kMode>, DH>::kFloats) * sizeof(float);
    const dim3 grid_q((unsigned)xcd_sub_grid(max_q_tiles * p.num_heads, kF32Split)), grid_k((unsigned)xcd_sub_grid(max_k_tiles * p.num_heads, kF32KeySplit)), block(kThreads);
    if constexpr (kMode != kF32Far) {
      if (p.laid.base && !p.fp32_products) {
        static std::atomic<uint64_t> laid_lds_done{0};
        const hipError_t r = raise_lds_limit(&bwd_dkv_f32_kernel<DH, kMode, true>, laid_lds_done, dev, lds_bytes);
        if (r != hipSuccess) return r;
        const dim3 grid((unsigned)xcd_sub_grid(max_q_tiles * p.num_heads, 2));
        hipLaunchKernelGGL((lay_f32_kernel<DH, kMode, true>), grid, block, 0, stream, p);
        hipLaunchKernelGGL((bwd_dq_f32_kernel<DH, kMode, true>), grid_q, block, 0, stream, p);
        hipLaunchKernelGGL((lay_f32_kernel<DH, kMode, false>), grid, block, 0, stream, p);
        hipLaunchKernelGGL((bwd_dkv_f32_kernel<DH, kMode, true>), grid_k, block, lds_bytes, stream, p);
        return hipGetLastError();
      }
    }
    static std::atomic<uint64_t> lds_done{0};
    const hipError_t r = raise_lds_limit(&bwd_dkv_f32_kernel<DH, kMode, false>, lds_done, dev, lds_bytes);
    if (r != hipSuccess) return r;
    hipLaunchKernelGGL((bwd_dq_f32_kernel<DH, kMode, false>), grid_q, block, 0, stream, p);
    hipLaunchKernelGGL((bwd_dkv_f32_kernel<DH, kMode, false>), grid_k, block, lds_bytes, stream, p);
    return hipGetLastError();
  });
}

}  // namespace sba
