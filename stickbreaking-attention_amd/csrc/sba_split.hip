// The 16-bit kernels for problems too small to fill the chip with workgroups of 128 query rows (or of a key tile).
//
// What bounds such a problem is the time one workgroup needs for its longest row: a wave takes ~0.5 us per 32 keys however
// empty the chip is.  So a workgroup's four waves work on the SAME 32 query rows (forward, dQ) and split the keys, or on the same
// 32 keys (dK/dV) and split the rows.  Four times the workgroups, a quarter of the steps each; the partial sums of the waves are
// added through LDS at the end, in a fixed order.  The price is that K and V (Q and dO) are staged per 32 rows instead of per 128,
// which is why these kernels stop paying once the chip is full (the rule stands with the launches).
//
// A wave stages the 32 keys (rows) it works on for itself, so nothing waits for another wave's loads.  Forward: a wave takes a
// contiguous part of the keys and starts from a product of 1; what the waves above have left of the stick is multiplied on at the end (into
// the sums, and into the recorded products).  dQ: C below a sub-tile is a sum with signs that is rounded with the weights, so the waves take
// every fourth sub-tile and exchange one number per row and step, with one barrier.  dK/dV: nothing is exchanged.  Against staging together with
// three barriers per step of 128 keys, us: forward, 1 head x 2048 tokens x 64 19.6 -> 16.2, 4096 36.2 -> 27.9; head_dim 50, 4096 53.6 -> 41.9; training
// pass of 7 heads, 8191 tokens in 14 sequences of up to 1886, head_dim 50 180 -> 172, 64 135 -> 129.
#include "sba_device.hpp"
#include "sba_host.hpp"
#include "sba_params.hpp"
#include "sba_sched.hpp"

#include <type_traits>

namespace sba {

constexpr int kSplitRows = 32;                            // query rows (or keys) per workgroup
constexpr int kSplitSubs = kBlockQ / kSplitRows;          // workgroups per 128-row tile of the schedule
constexpr int kStep = 128;                                // keys (or rows) per step

// The waves' partial results of a 32 x DH block, summed and written: acc[dt][r] is row 8*(r/4) + 4*half + r%4, column
// 32*dt + col.  `add` (or NULL): rows whose multiples add_scale[row] are added.
template <typename T, int DH, int kLoad>
__device__ __forceinline__ void reduce_store(float* lds, const f32x16 (&acc)[DH / 32], float scale, T* out, int64_t stride, int rows, int D,
                                             const T* add = nullptr, int64_t add_stride = 0, const float* add_scale = nullptr) {
  constexpr int kStride = DH + 4, kPer = 32 * DH / kThreads;      // consecutive columns per thread
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, half = lane >> 5, col = lane & 31;
  __syncthreads();
#pragma unroll
  for (int dt = 0; dt < DH / 32; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) lds[(wave * 32 + 8 * (r >> 2) + 4 * half + (r & 3)) * kStride + 32 * dt + col] = acc[dt][r];
  __syncthreads();
  const int row = threadIdx.x / (DH / kPer), c0 = (threadIdx.x % (DH / kPer)) * kPer;
  if (row >= rows) return;
  float x[kPer];
#pragma unroll
  for (int i = 0; i < kPer; i += 4) {
    f32x4 sum = *reinterpret_cast<const f32x4*>(lds + row * kStride + c0 + i);
#pragma unroll
    for (int w = 1; w < kWaves; w++) {
      const f32x4 y = *reinterpret_cast<const f32x4*>(lds + (w * 32 + row) * kStride + c0 + i);
#pragma unroll
      for (int k = 0; k < 4; k++) sum[k] += y[k];
    }
#pragma unroll
    for (int k = 0; k < 4; k++) x[i + k] = sum[k] * scale;
  }
  if (add) {
#pragma unroll
    for (int i = 0; i < kPer; i++)
      if (kLoad == kLoadAligned || c0 + i < D) x[i] += add_scale[row] * (float)add[row * add_stride + c0 + i];
  }
  T* o = out + row * stride + c0;
  if (kLoad == kLoadAligned) {
#pragma unroll
    for (int i = 0; i < kPer; i += 8)
      *reinterpret_cast<u32x4*>(o + i) = u32x4{pack2<T>(x[i], x[i + 1]), pack2<T>(x[i + 2], x[i + 3]), pack2<T>(x[i + 4], x[i + 5]),
                                               pack2<T>(x[i + 6], x[i + 7])};
  } else {
#pragma unroll
    for (int i = 0; i < kPer; i++)
      if (c0 + i < D) o[i] = (T)x[i];
  }
}

template <int DH> struct SplitLds {
  static constexpr int kSub = 32 * lds_stride<DH>();                                  // elements of a wave's part of one staged tensor
  static constexpr size_t kStage = (size_t)2 * kWaves * kSub * 2, kSums = (size_t)kWaves * 32 * (DH + 4) * 4;
  static constexpr size_t kBytes = kStage > kSums ? kStage : kSums;
};

// What the lanes of a wave hand each other through LDS of the wave's own needs no barrier, only the order of the accesses.
__device__ __forceinline__ void wave_fence() { asm volatile("" ::: "memory"); }

// S^T (or dP^T) of a 32-row operand in registers against the 32 rows `rows` of a staged tile.
template <typename T, int DH>
__device__ __forceinline__ f32x16 scores32(const T* rows, const typename Elem<T>::vec8 (&x)[DH / 16], int krow, int half) {
  constexpr int kSteps = DH / 16;
  f32x16 s;
#pragma unroll
  for (int r = 0; r < 16; r++) s[r] = 0.f;
  typename Elem<T>::vec8 a[kSteps];
#pragma unroll
  for (int kk = 0; kk < kSteps; kk++) a[kk] = lds_row8<T>(rows, lds_stride<DH>(), krow, 16 * kk + 8 * half);
#pragma unroll
  for (int kk = 0; kk < kSteps; kk++) s = Elem<T>::mfma(a[kk], x[kk], s);
  return s;
}

// acc[dt] += w . rows, contracted over the 32 staged rows; w: 16 packed weights per lane (row 16*half + r).
template <typename T, int DH>
__device__ __forceinline__ void contract32(f32x16 (&acc)[DH / 32], const uint32_t (&w)[8], const T* rows, int half, int lane) {
#pragma unroll
  for (int c = 0; c < 2; c++) {
    const typename Elem<T>::vec8 a = as_vec8<T>(u32x4{w[4 * c], w[4 * c + 1], w[4 * c + 2], w[4 * c + 3]});
#pragma unroll
    for (int dt = 0; dt < DH / 32; dt++)
      acc[dt] = Elem<T>::mfma(a, lds_col8<T>(rows, lds_stride<DH>(), 16 * half + 8 * c, 32 * dt, lane), acc[dt]);
  }
}

// kCarryOnly: as in fwd_kernel, and with this kernel's products bit for bit.
template <typename T, int DH, int kLoad, bool kCarryOnly>
__global__ __launch_bounds__(kThreads, 2) void fwd_split_kernel(FwdParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  __shared__ __attribute__((aligned(16))) float xch[kWaves][32];
  __shared__ float rem_lds[32];
  if (!kCarryOnly && (int)blockIdx.x < p.sched.service) {
    forward_service(p.sched, blockIdx.x);
    return;
  }
  const int wg = blockIdx.x - p.sched.service;
  int head, slot, sub;
  xcd_head_tile_sub(wg, kSplitSubs, p.num_heads, &head, &slot, &sub);
  Tile tile;
  int64_t r0, r1;
  if (!forward_tile(p, slot, sub, kSplitRows, &tile, &r0, &r1)) {
    if (!kCarryOnly && r0 < r1) {      // rows of no sequence: o = rem = 0
      zero_rows<T>(p.o, head, r0, r1, p.head_dim);
      for (int64_t r = r0 + threadIdx.x; r < r1; r += kThreads) {
        ((T*)p.rem.ptr)[head * p.rem.sh + r * p.rem.st] = (T)0;
        p.row_stat[head * p.stat_sh + r] = 0.f;
      }
    }
    return;
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, col = lane & 31;
  const int L = tile.seq_len, ac = p.attend_current, D = kLoad == kLoadPadded ? p.head_dim : DH;
  const int q0 = tile.origin + sub * kSplitRows;
  if (q0 >= L) return;
  const int64_t tok0 = tile.seq_start;
  const T* qb = (const T*)p.q.ptr + tile.seq_id * p.q.sb + head * p.q.sh + tok0 * p.q.st;
  const T* kb = (const T*)p.k.ptr + tile.seq_id * p.k.sb + head * p.k.sh + tok0 * p.k.st;
  const T* vb = (const T*)p.v.ptr + tile.seq_id * p.v.sb + head * p.v.sh + tok0 * p.v.st;
  const int qi = q0 + col;
  const int n_qt = (L + kBlockQ - 1) / kBlockQ;
  float* carry = p.carry ? p.carry + (int64_t)head * p.carry_head_stride + tile.carry_base + sub * kSplitRows : nullptr;
  const int last_key = min(q0 + kSplitRows, L) - 2 + ac, n_sub = last_key < 0 ? 0 : last_key / 32 + 1;
  const int krow = mfma_row_to_key32(col);
  auto carry_row = [&](int u) { return carry + carry_offset(u, n_qt) + (tile.origin - kBlockQ * (u >> 2)); };
  // (Recorded in whole groups of four: the kernels that sweep 64 keys read the upper sub-tile of a pair.)
  if (carry && wave == 0 && half == 0)
    for (int u = n_sub; u & 3; u++) carry_row(u)[col] = 1.f;

  // This wave's sub-tiles, the last wave's the uppermost: swept on their own, downwards from a product of 1.  The parts are cut by where the rows
  // lie and not by how many the sequence has (of which one less may see a key of the last sub-tile), so that no row's bits depend on the next.
  const int q_sub = q0 / 32, per = q_sub / kWaves + 1, end = q_sub + 1 - (kWaves - 1 - wave) * per, top = min(end, n_sub), bottom = max(end - per, 0);
  T* const k_lds = reinterpret_cast<T*>(lds_raw) + wave * (2 * SplitLds<DH>::kSub);
  T* const v_lds = k_lds + SplitLds<DH>::kSub;
  const RowSource<T> ksrc = make_row_source<T, kLoad>(kb, p.k.st, L, D), vsrc = make_row_source<T, kLoad>(vb, p.v.st, L, D);
  TileCopy<T, DH, 32, kLoad, 64> ck, cv;
  if (top > bottom) {
    ck.load(ksrc, (top - 1) * 32);
    if (!kCarryOnly) cv.load(vsrc, (top - 1) * 32);
  }
  typename Elem<T>::vec8 qf[DH / 16];
  load_operand<T, kLoad>(qf, make_row_source<T, kLoad>(qb, p.q.st, L, D), qi, half);
  f32x16 oacc[DH / 32];
#pragma unroll
  for (int dt = 0; dt < DH / 32; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) oacc[dt][r] = 0.f;
  float prod = 1.f;      // product over the keys of this wave's sub-tiles done so far
  settle(qf);
  float* const lowest_row = carry_row(bottom);
  float* row = carry_row(top - 1);
  for (int u = top - 1; u >= bottom; --u) {
    const int j0 = 32 * u;
    ck.store(k_lds);
    if (!kCarryOnly) cv.store(v_lds);
    wave_fence();
    if (u > bottom) {
      ck.load(ksrc, j0 - 32);
      if (!kCarryOnly) cv.load(vsrc, j0 - 32);
    }
    f32x16 s[1];
    s[0] = scores32<T, DH>(k_lds, qf, krow, half);
    Weights<16> w;
    const int lim = qi + ac - j0 - 16 * half;
    if (j0 + 31 > q0 - 1 + ac) w.template front<true>(s, p.scale_log2, lim); else w.template front<false>(s, p.scale_log2, lim);
    const float oth = other_half(w.run, half);
    if (carry && half == 0) row[col] = prod;
    row -= carry_step(u - 1, n_qt);
    const float seed = half ? prod : prod * oth;              // the upper half-wave holds the higher keys
    prod *= w.run * oth;
    if (!kCarryOnly) {
      w.back(seed);
      uint32_t pk[8];
#pragma unroll
      for (int i = 0; i < 8; i++) pk[i] = pack2<T>(w.t[2 * i], w.t[2 * i + 1]);
      contract32<T, DH>(oacc, pk, v_lds, half, lane);
    }
    wave_fence();
  }
  // Below the sub-tiles of the waves above: their products come on top.
  if (half == 0) xch[wave][col] = prod;
  __syncthreads();
  float above = 1.f;
  prod = 1.f;
#pragma unroll
  for (int x = kWaves - 1; x >= 0; --x) {
    if (x == wave) above = prod;
    prod *= xch[x][col];
  }
  if (carry && half == 0 && wave < kWaves - 1) {
    // (Four under way at a time: one after the other, 15 sub-tiles took as many latencies.)
    row = lowest_row;
    int u = bottom;
    for (; u + 4 <= top; u += 4) {
      float* at[4];
      float x[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        at[i] = row;
        x[i] = row[col];
        row += carry_step(u + i, n_qt);
      }
#pragma unroll
      for (int i = 0; i < 4; i++) at[i][col] = x[i] * above;
    }
    for (; u < top; u++) {
      row[col] *= above;
      row += carry_step(u, n_qt);
    }
  }
  if (kCarryOnly) return;
  if (wave < kWaves - 1) {
#pragma unroll
    for (int g = 0; g < 4; g++) {
      f32x4 scale = {1.f, 1.f, 1.f, 1.f};      // of rows 8 g + 4 half ..
#pragma unroll
      for (int x = kWaves - 1; x > 0; --x)
        if (x > wave) scale *= *reinterpret_cast<const f32x4*>(&xch[x][8 * g + 4 * half]);
#pragma unroll
      for (int dt = 0; dt < DH / 32; dt++)
#pragma unroll
        for (int r = 0; r < 4; r++) oacc[dt][4 * g + r] *= scale[r];
    }
  }
  if (wave == 0 && half == 0) {
    rem_lds[col] = prod;
    if (qi < L) {
      ((T*)p.rem.ptr)[tile.seq_id * p.rem.sb + head * p.rem.sh + (tok0 + qi) * p.rem.st] = (T)prod;
      p.row_stat[tile.seq_id * p.stat_sb + head * p.stat_sh + tok0 + qi] = fast_log2(prod);
    }
  }
  T* ob = (T*)p.o.ptr + tile.seq_id * p.o.sb + head * p.o.sh + (tok0 + q0) * p.o.st;
  reduce_store<T, DH, kLoad>(reinterpret_cast<float*>(lds_raw), oacc, 1.f, ob, p.o.st, L - q0, D,
                             p.add_rem ? vb + (int64_t)q0 * p.v.st : nullptr, p.v.st, rem_lds);
}

template <typename T, int DH, int kLoad>
__global__ __launch_bounds__(kThreads, DH == 128 ? 1 : 2) void bwd_dq_split_kernel(BwdParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  __shared__ float xch[2][kWaves][32];
  int head, slot, sub;
  xcd_head_tile_sub(blockIdx.x, kSplitSubs, p.num_heads, &head, &slot, &sub);
  if (slot >= p.counts[kCountQ]) {
    int64_t r0, r1;
    if (uncovered_rows(p.counts, slot, p.total_tokens, sub, kSplitRows, &r0, &r1)) {      // rows of no sequence: zero gradients
      zero_rows<T>(p.dq, head, r0, r1, p.head_dim);
      zero_rows<T>(p.dk, head, r0, r1, p.head_dim);
      zero_rows<T>(p.dv, head, r0, r1, p.head_dim);
    }
    return;
  }
  const Tile tile = p.q_tiles[slot];
  if (p.tiny && tile.seq_len <= kTinyRows) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, col = lane & 31;
  const int L = tile.seq_len, ac = p.attend_current, D = kLoad == kLoadPadded ? p.head_dim : DH;
  const int q0 = tile.origin + sub * kSplitRows;
  if (q0 >= L) return;
  const int64_t tok0 = tile.seq_start;
  const T* qb = (const T*)p.q.ptr + tile.seq_id * p.q.sb + head * p.q.sh + tok0 * p.q.st;
  const T* kb = (const T*)p.k.ptr + tile.seq_id * p.k.sb + head * p.k.sh + tok0 * p.k.st;
  const T* vb = (const T*)p.v.ptr + tile.seq_id * p.v.sb + head * p.v.sh + tok0 * p.v.st;
  const T* dob = (const T*)p.d_o.ptr + tile.seq_id * p.d_o.sb + head * p.d_o.sh + tok0 * p.d_o.st;
  const int qi = q0 + col;
  const bool row_ok = qi < L;
  const int last_key = min(q0 + kSplitRows, L) - 2 + ac, n_kt = last_key < 0 ? 0 : last_key / kStep + 1;
  const int krow = mfma_row_to_key32(col);
  const int n_qt = (L + kBlockQ - 1) / kBlockQ;
  int64_t slot_row = (int64_t)head * p.carry_head_stride + tile.carry_base + sub * kSplitRows + carry_offset(wave, n_qt) + tile.origin;      // of this wave's sub-tile

  T* const k_lds = reinterpret_cast<T*>(lds_raw) + wave * (2 * SplitLds<DH>::kSub);
  T* const v_lds = k_lds + SplitLds<DH>::kSub;
  const RowSource<T> ksrc = make_row_source<T, kLoad>(kb, p.k.st, L, D), vsrc = make_row_source<T, kLoad>(vb, p.v.st, L, D);
  TileCopy<T, DH, 32, kLoad, 64> ck, cv;
  float n_prod = 1.f;      // the forward's product above this wave's sub-tile of the next step
  if (n_kt > 0) {
    ck.load(ksrc, 32 * wave);
    cv.load(vsrc, 32 * wave);
    if (32 * wave <= last_key) n_prod = (p.carry + slot_row)[col];
  }
  typename Elem<T>::vec8 qf[DH / 16], dof[DH / 16];
  load_operand<T, kLoad>(qf, make_row_source<T, kLoad>(qb, p.q.st, L, D), qi, half);
  load_operand<T, kLoad>(dof, make_row_source<T, kLoad>(dob, p.d_o.st, L, D), qi, half);
  float drem = 0.f;
  if (row_ok && p.d_rem.ptr) drem = (float)((const T*)p.d_rem.ptr)[tile.seq_id * p.d_rem.sb + head * p.d_rem.sh + (tok0 + qi) * p.d_rem.st];
  if (p.add_rem) {
    // The forward wrote o + rem * v: the gradient reaching rem is d_rem + d_o . v_i.
    float dot = 0.f;
    typename Elem<T>::vec8 vf[DH / 16];
    load_operand<T, kLoad>(vf, vsrc, qi, half);
#pragma unroll
    for (int kk = 0; kk < DH / 16; kk++)
#pragma unroll
      for (int t = 0; t < 8; t++) dot = fmaf((float)dof[kk][t], (float)vf[kk][t], dot);
    drem += dot + other_half(dot, half);
  }
  if (wave == 0 && half == 0 && row_ok) p.drem_eff[tile.seq_id * p.drem_sb + head * p.stat_sh + tok0 + qi] = drem;

  f32x16 dqacc[DH / 32];
#pragma unroll
  for (int dt = 0; dt < DH / 32; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) dqacc[dt][r] = 0.f;
  float prefix = 0.f;      // sum of g over the keys of the steps done so far
  settle(qf);
  settle(dof);
  settle(drem);
  for (int jt = 0; jt < n_kt; ++jt) {
    const int u = 4 * jt + wave, j0 = 32 * u;                 // this wave's sub-tile
    const bool active = j0 <= last_key;
    wave_fence();
    ck.store(k_lds);
    cv.store(v_lds);
    wave_fence();
    const float prod_in = n_prod;
    float* const prefix_row = p.prefix + slot_row;
    slot_row += carry_step4(u, n_qt);
    if (jt + 1 < n_kt) {
      ck.load(ksrc, j0 + kStep);
      cv.load(vsrc, j0 + kStep);
      if (j0 + kStep <= last_key) n_prod = (p.carry + slot_row)[col];
    }
    BwdMath<16> m;
    m.tot = m.oth_g = 0.f;
    if (active) {
      f32x16 s[1], dp[1];
      s[0] = scores32<T, DH>(k_lds, qf, krow, half);
      dp[0] = scores32<T, DH>(v_lds, dof, krow, half);
      const int lim = row_ok ? qi + ac - j0 - 16 * half : 0;
      if (j0 + 31 > q0 - 1 + ac || q0 + 31 >= L) bwd_math_front<1, true, false>(m, s, dp, p.scale_log2, lim, half, drem, prod_in);
      else bwd_math_front<1, false, false>(m, s, dp, p.scale_log2, lim, half, drem, prod_in);
    }
    if (half == 0) xch[jt & 1][wave][col] = m.tot + m.oth_g;
    lds_barrier();
    float below = prefix;
#pragma unroll
    for (int x = 0; x < kWaves; x++) {
      const float y = xch[jt & 1][x][col];
      if (x < wave) below += y;
      prefix += y;
    }
    if (active) {
      if (half == 0) prefix_row[col] = below;                 // C just below the sub-tile, for the dK/dV kernel
      uint32_t pk[8], dzk[8];
      bwd_math_back<T, 16, false>(m, below + (half ? m.oth_g : 0.f), pk, dzk);
      contract32<T, DH>(dqacc, dzk, k_lds, half, lane);
    }
  }
  T* dqb = (T*)p.dq.ptr + tile.seq_id * p.dq.sb + head * p.dq.sh + (tok0 + q0) * p.dq.st;
  reduce_store<T, DH, kLoad>(reinterpret_cast<float*>(lds_raw), dqacc, p.logit_scale, dqb, p.dq.st, L - q0, D);
}

// dK/dV, head_dim up to 64: 32 keys per workgroup, K and V stationary in registers.  Wave w takes every fourth group of 32 rows from the
// w-th on, counted from the group of the first row that sees the keys.
constexpr int kPzStride = 40;      // elements per row of a wave's P and dZ scratch
template <typename T, int kLoad>
__global__ __launch_bounds__(kThreads, 2) void bwd_dkv_split_kernel(BwdParams p) {
  constexpr int DH = 64, kStride = lds_stride<DH>();
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  __shared__ __attribute__((aligned(16))) T pz_lds[kWaves][2][32 * kPzStride];
  __shared__ float rem_lds[32];
  constexpr int subs = kBlockK / kSplitRows;
  int head, slot, sub;
  xcd_head_tile_sub(blockIdx.x, subs, p.num_heads, &head, &slot, &sub);
  if (slot >= p.counts[kCountK]) return;
  const Tile tile = p.k_tiles[slot];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, col = lane & 31;
  const int L = tile.seq_len, ac = p.attend_current, D = kLoad == kLoadPadded ? p.head_dim : DH;
  const int k0 = tile.origin + sub * kSplitRows;
  if (k0 >= L) return;
  const int64_t tok0 = tile.seq_start;
  const T* qb = (const T*)p.q.ptr + tile.seq_id * p.q.sb + head * p.q.sh + tok0 * p.q.st;
  const T* kb = (const T*)p.k.ptr + tile.seq_id * p.k.sb + head * p.k.sh + tok0 * p.k.st;
  const T* vb = (const T*)p.v.ptr + tile.seq_id * p.v.sb + head * p.v.sh + tok0 * p.v.st;
  const T* dob = (const T*)p.d_o.ptr + tile.seq_id * p.d_o.sb + head * p.d_o.sh + tok0 * p.d_o.st;
  const int64_t n_qt = (L + kBlockQ - 1) / kBlockQ;
  const int u = k0 >> 5;
  const int64_t slot0 = (int64_t)head * p.carry_head_stride + tile.carry_base + carry_offset(u, n_qt) - kBlockQ * (u >> 2);
  const float* carry = p.carry + slot0;
  const float* prefix = p.prefix + slot0;
  const float* drem_plane = p.drem_eff + tile.seq_id * p.drem_sb + head * p.stat_sh + tok0;
  const int first_row = k0 + 1 - ac;                          // first row that sees key k0
  const int i_first = first_row / 32 + wave, i_end = first_row < L ? (L + 31) / 32 : 0;      // this wave's groups of 32 rows: every fourth

  const RowSource<T> qsrc = make_row_source<T, kLoad>(qb, p.q.st, L, D), dosrc = make_row_source<T, kLoad>(dob, p.d_o.st, L, D);
  T* const q_lds = reinterpret_cast<T*>(lds_raw) + wave * (2 * SplitLds<DH>::kSub);
  T* const do_lds = q_lds + SplitLds<DH>::kSub;
  TileCopy<T, DH, 32, kLoad, 64> cq, cdo;
  float n_prod = 1.f, n_prefix = 0.f, n_drem = 0.f;
  auto fetch_rows = [&](int i) {
    const int qi = 32 * i + col;
    cq.load(qsrc, 32 * i);
    cdo.load(dosrc, 32 * i);
    n_prod = carry[qi];
    n_prefix = prefix[qi];
    n_drem = qi < L ? drem_plane[qi] : 0.f;
  };
  if (i_first < i_end) fetch_rows(i_first);
  const int key = k0 + mfma_row_to_key32(col);
  typename Elem<T>::vec8 kf[DH / 16], vf[DH / 16];
  load_operand<T, kLoad>(kf, make_row_source<T, kLoad>(kb, p.k.st, L, D), key, half);
  load_operand<T, kLoad>(vf, make_row_source<T, kLoad>(vb, p.v.st, L, D), key, half);
  f32x16 dkacc[DH / 32], dvacc[DH / 32];
#pragma unroll
  for (int dt = 0; dt < DH / 32; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) { dkacc[dt][r] = 0.f; dvacc[dt][r] = 0.f; }
  settle(kf);
  settle(vf);
  for (int i = i_first; i < i_end; i += kWaves) {
    wave_fence();
    cq.store(q_lds);
    cdo.store(do_lds);
    wave_fence();
    const float prod_in = n_prod, prefix_in = n_prefix, drem = n_drem;
    if (i + kWaves < i_end) fetch_rows(i + kWaves);
    const int w_first = 32 * i, w_last = w_first + 31, qi = w_first + col;
    f32x16 s[1], dp[1];
#pragma unroll
    for (int r = 0; r < 16; r++) { s[0][r] = 0.f; dp[0][r] = 0.f; }
    typename Elem<T>::vec8 b[DH / 16];
#pragma unroll
    for (int kk = 0; kk < DH / 16; kk++) b[kk] = lds_row8<T>(q_lds, kStride, col, 16 * kk + 8 * half);
#pragma unroll
    for (int kk = 0; kk < DH / 16; kk++) s[0] = Elem<T>::mfma(kf[kk], b[kk], s[0]);
#pragma unroll
    for (int kk = 0; kk < DH / 16; kk++) b[kk] = lds_row8<T>(do_lds, kStride, col, 16 * kk + 8 * half);
#pragma unroll
    for (int kk = 0; kk < DH / 16; kk++) dp[0] = Elem<T>::mfma(vf[kk], b[kk], dp[0]);
    uint32_t pk[8], dzk[8];
    float prod_lower, prefix_upper, prefix_next;
    bwd_tile_math<T, 1>(s, dp, p.scale_log2, k0 + 31 > w_first - 1 + ac || w_last >= L, qi < L ? qi + ac - k0 - 16 * half : 0, half, drem,
                        prod_in, prefix_in, pk, dzk, prod_lower, prefix_upper, prefix_next);
    // To a lane per key (wave-private): [row][key], this lane's 16 consecutive keys in row `col`.
    T* p_rows = pz_lds[wave][0];
    T* z_rows = pz_lds[wave][1];
#pragma unroll
    for (int c = 0; c < 2; c++) {
      *reinterpret_cast<u32x4*>(p_rows + col * kPzStride + 16 * half + 8 * c) = u32x4{pk[4 * c], pk[4 * c + 1], pk[4 * c + 2], pk[4 * c + 3]};
      *reinterpret_cast<u32x4*>(z_rows + col * kPzStride + 16 * half + 8 * c) = u32x4{dzk[4 * c], dzk[4 * c + 1], dzk[4 * c + 2], dzk[4 * c + 3]};
    }
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const int row0 = 16 * c + 8 * half;
      const typename Elem<T>::vec8 ap = lds_col8<T>(p_rows, kPzStride, row0, 0, lane), az = lds_col8<T>(z_rows, kPzStride, row0, 0, lane);
#pragma unroll
      for (int dt = 0; dt < DH / 32; dt++) {
        dvacc[dt] = Elem<T>::mfma(ap, lds_col8<T>(do_lds, kStride, row0, 32 * dt, lane), dvacc[dt]);
        dkacc[dt] = Elem<T>::mfma(az, lds_col8<T>(q_lds, kStride, row0, 32 * dt, lane), dkacc[dt]);
      }
    }
  }
  if (p.add_rem && threadIdx.x < 32 && k0 + (int)threadIdx.x < L)      // the forward wrote o + rem * v: dv_i gains rem_i * d_o_i
    rem_lds[threadIdx.x] = fast_exp2(p.row_stat[tile.seq_id * p.stat_sb + head * p.stat_sh + tok0 + k0 + threadIdx.x]);
  T* dvb = (T*)p.dv.ptr + tile.seq_id * p.dv.sb + head * p.dv.sh + (tok0 + k0) * p.dv.st;
  T* dkb = (T*)p.dk.ptr + tile.seq_id * p.dk.sb + head * p.dk.sh + (tok0 + k0) * p.dk.st;
  float* sums = reinterpret_cast<float*>(lds_raw);
  reduce_store<T, DH, kLoad>(sums, dvacc, 1.f, dvb, p.dv.st, L - k0, D, p.add_rem ? dob + (int64_t)k0 * p.d_o.st : nullptr, p.d_o.st, rem_lds);
  reduce_store<T, DH, kLoad>(sums, dkacc, p.logit_scale, dkb, p.dk.st, L - k0, D);
}

// f(element type, width, load) for the 16-bit types.
template <typename F>
static hipError_t by_shape(int dtype_is_f16, int head_dim, int load, F&& f) {
  auto with = [&](auto t) {
    auto wide = [&](auto dh) {
      return load == kLoadAligned ? f(t, dh, std::integral_constant<int, kLoadAligned>()) : f(t, dh, std::integral_constant<int, kLoadPadded>());
    };
    return head_dim > 64 ? wide(std::integral_constant<int, 128>()) : wide(std::integral_constant<int, 64>());
  };
  return dtype_is_f16 ? with(_Float16()) : with((__bf16)0.f);
}

template <typename Kernel, typename Params>
static hipError_t launch_split(Kernel kernel, std::atomic<uint64_t>& lds_done, size_t lds_bytes, unsigned wgs, const Params& p, hipStream_t stream) {
  int dev = 0, cus = 0;
  hipError_t e = device_cus(&dev, &cus);
  if (e == hipSuccess) e = raise_lds_limit(kernel, lds_done, dev, lds_bytes);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3(wgs), dim3(kThreads), lds_bytes, stream, p);
  return hipGetLastError();
}

template <bool kCarryOnly>
static hipError_t launch_fwd_split_t(const FwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream) {
  return by_shape(dtype_is_f16, p.head_dim, p.load, [&](auto t, auto dh, auto load) {
    static std::atomic<uint64_t> lds_done{0};
    return launch_split(&fwd_split_kernel<decltype(t), decltype(dh)::value, decltype(load)::value, kCarryOnly>, lds_done,
                        SplitLds<decltype(dh)::value>::kBytes, (unsigned)(xcd_sub_grid(max_tiles * p.num_heads, kSplitSubs) + p.sched.service), p, stream);
  });
}
hipError_t launch_fwd_split(const FwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream) {
  return launch_fwd_split_t<false>(p, dtype_is_f16, max_tiles, stream);
}
hipError_t launch_fwd_split_carry_only(const FwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream) {
  return launch_fwd_split_t<true>(p, dtype_is_f16, max_tiles, stream);
}
hipError_t launch_bwd_dq_split(const BwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream) {
  return by_shape(dtype_is_f16, p.head_dim, p.load, [&](auto t, auto dh, auto load) {
    static std::atomic<uint64_t> lds_done{0};
    return launch_split(&bwd_dq_split_kernel<decltype(t), decltype(dh)::value, decltype(load)::value>, lds_done, SplitLds<decltype(dh)::value>::kBytes,
                        (unsigned)xcd_sub_grid(max_tiles * p.num_heads, kSplitSubs), p, stream);
  });
}
// max_tiles: key tiles of kBlockK keys; head_dim up to 64.
hipError_t launch_bwd_dkv_split(const BwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream) {
  return by_shape(dtype_is_f16, p.head_dim, p.load, [&](auto t, auto, auto load) {
    static std::atomic<uint64_t> lds_done{0};
    return launch_split(&bwd_dkv_split_kernel<decltype(t), decltype(load)::value>, lds_done, SplitLds<64>::kBytes,
                        (unsigned)xcd_sub_grid(max_tiles * p.num_heads, kBlockK / kSplitRows), p, stream);
  });
}

}  // namespace sba
