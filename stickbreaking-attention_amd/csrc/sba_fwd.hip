// Forward stick-breaking attention for gfx950.
//
// One workgroup = one tile of 128 query rows of one (head, sequence); wave w owns rows 32w..32w+31, lane l
// owns query l%32.  Key tiles of KT keys (32 on the head_dim 128 fast path, else 64) are swept in REVERSE from the
// causal diagonal (the order in which the stick is broken:
// stickbreaking_attention/sb_varlen/sb_varlen_fwd.py:155-165), so the running product
// prod_{j<k<i} (1 - sigma(z_ik)) is carried forward in registers and never has to be divided out.
//
// Per element, in linear space (base-2 exponentials, as sb_varlen_fwd.py:296 and softplus.py:8-12 do):
//     e = 2^x, x = z log2(e)          1 - sigma = 1/(1+e)          R_ij = prod_{j<=k<i} 1/(1+e_ik)
//     A_ij = sigma_ij R_i,j+1 = e_ij R_ij
// which needs one transcendental per element and one more per four (v_exp_f32, v_rcp_f32) where the log-space form
// log A = x - softplus2(x) + cumsum(-softplus2) needs three.  The product can only underflow where A itself is
// below 2^-126, and row_stat = log2(prod) is taken once per row at the end.
#include "sba_device.hpp"
#include "sba_dma.hpp"
#include "sba_params.hpp"
#include "sba_sched.hpp"

namespace sba {

// What a wave's rows come to: o (and the remainder's share of it), rem, row_stat.  oacc[dt][r]: query row 8*(r/4) + 4*half + r%4 of this
// wave, column 32*dt + col; prod: the remainder of row w_first + col.
template <typename T, int DH, int kLoad>
__device__ __forceinline__ void store_rows(const FwdParams& p, const Tile& tile, int head, int w_first, int half, int col, const T* vb,
                                           const f32x16 (&oacc)[DH / 32], float prod) {
  constexpr bool kFast = kLoad != kLoadScalar;
  // (Reading v a row at a time, a tile's 16 latencies took a tenth of the forward with the remainder: 211 us instead of 190, 16 heads x 128,
  // 16384 tokens; 122 and 111 us, 12 heads x 64.  Padded rows, 4 at a time over all columns, since 16 spill in the loop (187 us instead of 165, 12 heads x
  // 96): 12 heads, 20 x 500 tokens, head_dim 50 46 -> 39, 80 61 -> 50, 127 88 -> 67; 4 heads x 80, 8 x 52 13.8 -> 9.1; without the remainder, which pays
  // for one spilled register, 1.00 on average, up to 1.04 at 127.)
  constexpr bool kBatched = kLoad == kLoadAligned;
  constexpr int kDTiles = DH / 32;
  const int L = tile.seq_len, D = p.head_dim, qi = w_first + col;
  T* ob = (T*)p.o.ptr + tile.seq_id * p.o.sb + head * p.o.sh + (int64_t)tile.seq_start * p.o.st;
  if (p.add_rem) {
    // o + rem * v (the step callers of the reference apply to its outputs, tests/test_varlen.py:103): the row's
    // remainder is held by the lane whose query it is.
    if (kBatched) {      // 16 rows of v under way at a time
      const RowSink<T> sink = make_row_sink<T>(ob, p.o.st, L, D);
      const RowSource<T> vsrc = make_row_source<T, kLoad>(vb, p.v.st, L, D);
      const int voff = 4 * half * vsrc.stride_bytes + col * (int)sizeof(T), sbase = __builtin_amdgcn_readfirstlane(w_first * vsrc.stride_bytes);
      float rem_row[16];
#pragma unroll
      for (int r = 0; r < 16; r++) rem_row[r] = __shfl(prod, 8 * (r >> 2) + 4 * half + (r & 3));
#pragma unroll
      for (int dt = 0; dt < kDTiles; dt++) {
        f32x16 acc = oacc[dt];
        uint16_t v[16];
#pragma unroll
        for (int r = 0; r < 16; r++) v[r] = __builtin_amdgcn_raw_buffer_load_b16(vsrc.rsrc, voff, sbase + (8 * (r >> 2) + (r & 3)) * vsrc.stride_bytes + 64 * dt, 0);
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] += rem_row[r] * (float)__builtin_bit_cast(T, v[r]);
        store_acc_tile<T>(sink, acc, 1.f, w_first, 32 * dt, half, col, DH);
      }
    } else if (kFast) {      // 4 rows
      const RowSink<T> sink = make_row_sink<T>(ob, p.o.st, L, D);
      const RowSource<T> vsrc = make_row_source<T, kLoad>(vb, p.v.st, L, D);
      const int voff = 4 * half * vsrc.stride_bytes + col * (int)sizeof(T), sbase = __builtin_amdgcn_readfirstlane(w_first * vsrc.stride_bytes);
      f32x16 acc[kDTiles];
#pragma unroll
      for (int g = 0; g < 4; g++) {
        uint16_t v[4][kDTiles];
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
          for (int dt = 0; dt < kDTiles; dt++) v[r][dt] = __builtin_amdgcn_raw_buffer_load_b16(vsrc.rsrc, voff, sbase + (8 * g + r) * vsrc.stride_bytes + 64 * dt, 0);
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float rem_row = __shfl(prod, 8 * g + 4 * half + r);
#pragma unroll
          for (int dt = 0; dt < kDTiles; dt++) acc[dt][4 * g + r] = oacc[dt][4 * g + r] + rem_row * (float)__builtin_bit_cast(T, v[r][dt]);
        }
      }
#pragma unroll
      for (int dt = 0; dt < kDTiles; dt++) store_acc_tile<T>(sink, acc[dt], 1.f, w_first, 32 * dt, half, col, D);
    } else {
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int lr = 8 * (r >> 2) + 4 * half + (r & 3);
        const int row = w_first + lr;
        const float rem_row = __shfl(prod, lr);
#pragma unroll
        for (int dt = 0; dt < kDTiles; dt++) {
          const int d = 32 * dt + col;
          if (row < L && d < D)
            ob[(int64_t)row * p.o.st + d] = (T)(oacc[dt][r] + rem_row * (float)vb[(int64_t)row * p.v.st + d]);
        }
      }
    }
  } else if (kFast) {
    const RowSink<T> sink = make_row_sink<T>(ob, p.o.st, L, D);
#pragma unroll
    for (int dt = 0; dt < kDTiles; dt++) store_acc_tile<T>(sink, oacc[dt], 1.f, w_first, 32 * dt, half, col, kLoad == kLoadPadded ? D : DH);
  } else {
#pragma unroll
    for (int dt = 0; dt < kDTiles; dt++) {
      const int d = 32 * dt + col;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int row = w_first + 8 * (r >> 2) + 4 * half + (r & 3);
        if (row < L && d < D) ob[(int64_t)row * p.o.st + d] = (T)oacc[dt][r];
      }
    }
  }
  if (half == 0 && qi < L) {
    T* rb = (T*)p.rem.ptr + tile.seq_id * p.rem.sb + head * p.rem.sh + (int64_t)(tile.seq_start + qi) * p.rem.st;
    *rb = (T)prod;
    p.row_stat[tile.seq_id * p.stat_sb + head * p.stat_sh + tile.seq_start + qi] = fast_log2(prod);
  }
}

// kCarryOnly: only the products of (1 - sigma) above every sub-tile are rebuilt (into `carry`), for a backward whose
// forward did not keep them: no V, no P V, no outputs.
template <typename T, int DH, int kLoad, int KT, int kMinWaves, bool kCarryOnly = false>
__global__ __launch_bounds__(kThreads, kMinWaves) void fwd_kernel(FwdParams p) {
  constexpr bool kFast = kLoad != kLoadScalar;
  constexpr int NT = KT / 32;         // MFMA row tiles per key tile: a lane owns N = 16*NT consecutive keys
  constexpr int N = 16 * NT;
  typedef typename Elem<T>::vec8 vec8;
  constexpr int kRowStride = lds_stride<DH>();
  constexpr int kSteps = DH / 16;    // MFMA k-steps over head_dim
  constexpr int kDTiles = DH / 32;   // 32-wide output tiles over head_dim
  __shared__ __attribute__((aligned(16))) T k_lds[KT * kRowStride];
  __shared__ __attribute__((aligned(16))) T v_lds[KT * kRowStride];

  if (!kCarryOnly && (int)blockIdx.x < p.sched.service) {
    forward_service(p.sched, blockIdx.x);
    return;
  }
  int head, slot;
  xcd_head_tile(blockIdx.x - p.sched.service, p.num_heads, &head, &slot);
  Tile tile;
  int64_t r0, r1;
  if (!forward_tile(p, slot, 0, kBlockQ, &tile, &r0, &r1)) {
    if (!kCarryOnly && r0 < r1) {      // rows of no sequence: o = rem = 0
      zero_rows<T>(p.o, head, r0, r1, p.head_dim);
      for (int64_t r = r0 + threadIdx.x; r < r1; r += kThreads) {
        ((T*)p.rem.ptr)[head * p.rem.sh + r * p.rem.st] = (T)0;
        p.row_stat[head * p.stat_sh + r] = 0.f;
      }
    }
    return;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, half = lane >> 5, col = lane & 31;
  const int L = tile.seq_len, q0 = tile.origin, ac = p.attend_current, D = p.head_dim;

  const T* qb = (const T*)p.q.ptr + tile.seq_id * p.q.sb + head * p.q.sh + (int64_t)tile.seq_start * p.q.st;
  const T* kb = (const T*)p.k.ptr + tile.seq_id * p.k.sb + head * p.k.sh + (int64_t)tile.seq_start * p.k.st;
  const T* vb = (const T*)p.v.ptr + tile.seq_id * p.v.sb + head * p.v.sh + (int64_t)tile.seq_start * p.v.st;

  // This lane's query row as the B operand of S^T = K Q^T: 8 consecutive head_dim elements per k-step.
  const int qi = q0 + wave * 32 + col;
  vec8 qf[kSteps];
  load_operand<T, kLoad>(qf, make_row_source<T, kLoad>(qb, p.q.st, L, D), qi, half);

  const int last_row = min(q0 + kBlockQ, L) - 1;
  const int last_key = last_row - 1 + ac;                    // last key any row of this tile can see
  const int n_kt = last_key < 0 ? 0 : last_key / KT + 1;
  const int w_first = q0 + wave * 32, w_last = w_first + 31;   // this wave's rows

  f32x16 oacc[kDTiles];
#pragma unroll
  for (int dt = 0; dt < kDTiles; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) oacc[dt][r] = 0.f;
  float prod = 1.f;    // prod over the keys already swept of (1 - sigma): both half-waves hold the same value
  const int n_qt = (L + kBlockQ - 1) / kBlockQ;
  float* carry = p.carry ? p.carry + (int64_t)head * p.carry_head_stride + tile.carry_base : nullptr;

  const RowSource<T> ksrc = make_row_source<T, kLoad>(kb, p.k.st, L, D), vsrc = make_row_source<T, kLoad>(vb, p.v.st, L, D);
  TileCopy<T, DH, KT, kLoad> ck, cv;
  if (n_kt > 0) {
    ck.load(ksrc, (n_kt - 1) * KT);
    if (!kCarryOnly) cv.load(vsrc, (n_kt - 1) * KT);
  }
  // The recorded products are read per 64-key tile by the backward kernels that sweep 64 keys at a time, whichever
  // forward variant ran: a 32-key sweep that ends on the lower half of such a tile also records the (empty) product
  // above the upper half.
  // Slots of sub-tile u: a uniform base and this lane's row within the tile.
  const uint32_t lrow = wave * 32 + col;
  auto carry_row = [&](int u) { return carry + carry_offset(u, n_qt) + (q0 - kBlockQ * (u >> 2)); };
  if (NT == 1 && carry && half == 0 && (n_kt & 1)) carry_row(n_kt)[lrow] = 1.f;
  float* row_hi = carry_row(NT * n_kt - 1);                      // of the sub-tile at the upper edge of the tile
  for (int jt = n_kt - 1; jt >= 0; --jt) {
    const int j0 = jt * KT;
    __syncthreads();
    ck.store(k_lds);
    if (!kCarryOnly) cv.store(v_lds);
    __syncthreads();
    if (jt > 0) {
      const int jn = j0 - KT;
      ck.load(ksrc, jn);
      if (!kCarryOnly) cv.load(vsrc, jn);
    }
    // For the backward: the product over the keys between the upper 32-key sub-tile and the row, for every row
    // of the tile (the lower sub-tile's value follows once this tile's upper half is known).
    const int u_hi = NT * jt + NT - 1;                         // sub-tile at the upper edge of this tile
    float* const row_lo = NT == 2 ? row_hi - carry_step(u_hi - 1, n_qt) : row_hi;
    if (carry && half == 0) row_hi[lrow] = prod;
    row_hi = row_lo - carry_step(NT * jt - 1, n_qt);           // (for the next tile, if there is one)
    if (j0 > w_last - 1 + ac) {                               // nothing visible to this wave yet
      if (NT == 2 && carry && half == 0) row_lo[lrow] = prod;
      continue;
    }
    const bool diagonal = (j0 + KT - 1) > (w_first - 1 + ac);

    // The two MFMA phases of a step run at raised wave priority, the element-wise math at the default: a wave whose
    // next MFMA is ready then gets the issue port ahead of the other waves' vector-ALU streams (measured: -3 %).
    __builtin_amdgcn_s_setprio(3);
    // S^T tile: rows = keys (permuted so that a lane ends up with 32 consecutive keys), columns = queries.
    f32x16 s[NT];
#pragma unroll
    for (int mt = 0; mt < NT; mt++) {
#pragma unroll
      for (int r = 0; r < 16; r++) s[mt][r] = 0.f;
      const int krow = NT == 2 ? mfma_row_to_key(mt, col) : mfma_row_to_key32(col);
      if (NT == 1 && kFast) {
        // The K operands are requested four ahead of the MFMA that uses them: requested two at a time (what the
        // register allocator otherwise settles for) the wave pays the LDS latency four times per step.
        vec8 a[kSteps];
#pragma unroll
        for (int kk = 0; kk < 4; kk++) a[kk] = lds_row8<T>(k_lds, kRowStride, krow, 16 * kk + 8 * half);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < kSteps; kk++) {
          s[mt] = Elem<T>::mfma(a[kk], qf[kk], s[mt]);
          if (kk + 4 < kSteps) a[kk + 4] = lds_row8<T>(k_lds, kRowStride, krow, 16 * (kk + 4) + 8 * half);
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
#pragma unroll
        for (int kk = 0; kk < kSteps; kk++) {
          vec8 a = lds_row8<T>(k_lds, kRowStride, krow, 16 * kk + 8 * half);
          s[mt] = Elem<T>::mfma(a, qf[kk], s[mt]);
        }
      }
    }

    // This lane's N keys are j0 + N*half + R, R = 16*mt + r.
    __builtin_amdgcn_s_setprio(0);
    Weights<N> w;
    const int lim = qi + ac - j0 - N * half;                  // key R is visible iff R < lim
    if (diagonal) w.template front<true>(s, p.scale_log2, lim); else w.template front<false>(s, p.scale_log2, lim);
    const float run = w.run;
    const float oth = other_half(run, half);
    // The upper half-wave holds the higher keys, which come first in the sweep.
    const float seed = half ? prod : prod * oth;
    if (NT == 2 && carry && half == 0) row_lo[lrow] = seed;   // product above the lower sub-tile
    prod = (prod * oth) * run;
    if (kCarryOnly) continue;
    w.back(seed);
    __builtin_amdgcn_s_setprio(3);
    // O += P V: A = P from registers (k index <-> key 32*half + 8c + t), B = V gathered down the keys.
#pragma unroll
    for (int c = 0; c < KT / 16; c++) {
      u32x4 av;
#pragma unroll
      for (int i = 0; i < 4; i++) av[i] = pack2<T>(w.t[8 * c + 2 * i], w.t[8 * c + 2 * i + 1]);
      vec8 a = as_vec8<T>(av);
#pragma unroll
      for (int dt = 0; dt < kDTiles; dt++) {
        vec8 b = lds_col8<T>(v_lds, kRowStride, N * half + 8 * c, 32 * dt, lane);
        oacc[dt] = Elem<T>::mfma(a, b, oacc[dt]);
      }
    }
    __builtin_amdgcn_s_setprio(0);
  }

  if (kCarryOnly) return;
  store_rows<T, DH, kLoad>(p, tile, head, w_first, half, col, vb, oacc, prod);
}

// The same for aligned rows of 128 elements (kLoadAligned): key tiles of 32 keys come straight into LDS, one ahead of the tile that is
// worked on, in two buffers: no registers, no LDS writes and one barrier per tile instead of two.
// What bounds it: per 32 x 32 block 113 vector-ALU instructions (600 cycles) and 16 MFMAs (512 cycles), at three waves per SIMD, which
// keep one of the two pipes busy 94 % of the time and both 21 % (32 heads x 8 x 4096; 87 and 18 % on 25 sequences of up to 4096, whose
// diagonal tiles and ends weigh more); and the power limit (1.9 GHz).  32 heads x 8 x 4096: 1140 us with tiles through registers, 1100 here.  (head_dim 64 keeps its tiles of 64 keys: 107 us for 12 heads, 16384 tokens, against 112.)
template <typename T>
__global__ __launch_bounds__(kThreads, 3) void fwd_dma_kernel(FwdParams p) {
  typedef typename Elem<T>::vec8 vec8;
  constexpr int DH = 128, KT = 32, kSteps = DH / 16, kDTiles = DH / 32;
  constexpr int kPanel = KT * 64, kMat = kDTiles * kPanel, kBuf = 2 * kMat;      // bytes
  __shared__ __attribute__((aligned(16))) unsigned char lds_raw[2 * kBuf];
  lds_u8* const lds = (lds_u8*)lds_raw;
  const int lds_base = __builtin_amdgcn_readfirstlane((int)(uintptr_t)lds);

  if ((int)blockIdx.x < p.sched.service) {
    forward_service(p.sched, blockIdx.x);
    return;
  }
  int head, slot;
  xcd_head_tile(blockIdx.x - p.sched.service, p.num_heads, &head, &slot);
  Tile tile;
  int64_t r0, r1;
  if (!forward_tile(p, slot, 0, kBlockQ, &tile, &r0, &r1)) {
    if (r0 < r1) {      // rows of no sequence: o = rem = 0
      zero_rows<T>(p.o, head, r0, r1, p.head_dim);
      for (int64_t r = r0 + threadIdx.x; r < r1; r += kThreads) {
        ((T*)p.rem.ptr)[head * p.rem.sh + r * p.rem.st] = (T)0;
        p.row_stat[head * p.stat_sh + r] = 0.f;
      }
    }
    return;
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, col = lane & 31;
  const int L = tile.seq_len, q0 = tile.origin, ac = p.attend_current;
  const T* qb = (const T*)p.q.ptr + tile.seq_id * p.q.sb + head * p.q.sh + (int64_t)tile.seq_start * p.q.st;
  const T* kb = (const T*)p.k.ptr + tile.seq_id * p.k.sb + head * p.k.sh + (int64_t)tile.seq_start * p.k.st;
  const T* vb = (const T*)p.v.ptr + tile.seq_id * p.v.sb + head * p.v.sh + (int64_t)tile.seq_start * p.v.st;

  const int last_row = min(q0 + kBlockQ, L) - 1;
  const int last_key = last_row - 1 + ac;                    // last key any row of this tile can see
  const int n_kt = last_key < 0 ? 0 : last_key / KT + 1;
  const int w_first = q0 + wave * 32, w_last = w_first + 31, qi = w_first + col;

  // Tile jt into buffer jt & 1: waves 0 and 1 bring two panels of K each, 2 and 3 of V.  Row m is key mfma_row_to_key32(m): the MFMA's output row.
  const bool brings_v = wave >= 2;
  const int panel0 = 2 * (wave & 1), kv_st = (int)((brings_v ? p.v.st : p.k.st) * 2);
  const u32x4 desc = buffer_desc(brings_v ? vb : kb, (L - 1) * kv_st + 2 * DH);
  const int voff = mfma_row_to_key32(lane >> 2) * kv_st + panel0 * 64 + (((lane & 3) ^ ((lane >> 4) & 3)) << 4);
  auto request = [&](int jt) {
    const int soff = jt * KT * kv_st, dst = lds_base + (jt & 1) * kBuf + wave * (2 * kPanel);
#pragma unroll
    for (int i = 0; i < 2; i++) dma16x2<1024>(dst + i * kPanel, voff, desc, soff + 64 * i, soff + 64 * i + 8 * kv_st);
  };
  if (n_kt > 0) request(n_kt - 1);
  vec8 qf[kSteps];
  load_operand<T, kLoadAligned>(qf, make_row_source<T, kLoadAligned>(qb, p.q.st, L, DH), qi, half);

  f32x16 oacc[kDTiles];
#pragma unroll
  for (int dt = 0; dt < kDTiles; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) oacc[dt][r] = 0.f;
  float prod = 1.f;    // prod over the keys already swept of (1 - sigma): both half-waves hold the same value
  const int n_qt = (L + kBlockQ - 1) / kBlockQ;
  float* carry = p.carry ? p.carry + (int64_t)head * p.carry_head_stride + tile.carry_base : nullptr;
  // Slots of sub-tile u: a uniform base and this lane's row within the tile.  The products are read per 64 keys by backward kernels
  // that sweep as many at a time: a sweep that ends on the lower half also records the (empty) product above the upper half.
  const uint32_t lrow = wave * 32 + col;
  auto carry_row = [&](int u) { return carry + carry_offset(u, n_qt) + (q0 - kBlockQ * (u >> 2)); };
  if (carry && half == 0 && (n_kt & 1)) carry_row(n_kt)[lrow] = 1.f;
  float* row = carry_row(n_kt - 1);
  const int s15 = lane & 15, g = (lane >> 4) & 1;
  const int row_a = col * 64 + ((half ^ ((col >> 2) & 3)) << 4);                                                   // odd steps: ^ 32
  const int tr_k = (4 * half + (s15 >> 2)) * 64 + (((2 * g + ((s15 >> 1) & 1)) ^ half) << 4) + 8 * (s15 & 1);      // the next 4 rows: (^ 32) + 512
  vm_wait<0>();
  lds_barrier();
  for (int jt = n_kt - 1; jt >= 0; --jt) {
    const int j0 = jt * KT;
    if (jt > 0) request(jt - 1);
    if (carry && half == 0) row[lrow] = prod;                 // for the backward: the product over the keys between this tile and the row
    row -= carry_step(jt - 1, n_qt);
    if (j0 <= w_last - 1 + ac) {                              // (else nothing visible to this wave yet)
      const bool diagonal = (j0 + KT - 1) > (w_first - 1 + ac);
      lds_u8* kt = lds + (jt & 1) * kBuf;
      // The two MFMA phases of a step run at raised wave priority, the element-wise math at the default: a wave whose
      // next MFMA is ready then gets the issue port ahead of the other waves' vector-ALU streams.
      __builtin_amdgcn_s_setprio(3);
      f32x16 s[1];
#pragma unroll
      for (int r = 0; r < 16; r++) s[0][r] = 0.f;
      lds_u8* k0 = kt + row_a;
      lds_u8* k1 = kt + (row_a ^ 32);
      auto k_op = [&](int kk) { return lds_load<vec8>(((kk & 1) ? k1 : k0) + (kk >> 1) * kPanel); };
      vec8 a[4];
#pragma unroll
      for (int kk = 0; kk < 4; kk++) a[kk] = k_op(kk);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < kSteps; kk++) {
        s[0] = Elem<T>::mfma(a[kk & 3], qf[kk], s[0]);
        if (kk + 4 < kSteps) a[kk & 3] = k_op(kk + 4);
        __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_s_setprio(0);
      Weights<16> w;
      const int lim = qi + ac - j0 - 16 * half;               // key R is visible iff R < lim
      if (diagonal) w.template front<true>(s, p.scale_log2, lim); else w.template front<false>(s, p.scale_log2, lim);
      const float run = w.run;
      const float oth = other_half(run, half);
      const float seed = half ? prod : prod * oth;            // the upper half-wave holds the higher keys, which come first in the sweep
      prod = (prod * oth) * run;
      w.back(seed);
      __builtin_amdgcn_s_setprio(3);
      lds_u8* t0 = kt + kMat + tr_k;
      lds_u8* t1 = kt + kMat + (tr_k ^ 32) + 512;
#pragma unroll
      for (int c = 0; c < 2; c++) {
        u32x4 av;
#pragma unroll
        for (int i = 0; i < 4; i++) av[i] = pack2<T>(w.t[8 * c + 2 * i], w.t[8 * c + 2 * i + 1]);
#pragma unroll
        for (int dt = 0; dt < kDTiles; dt++)
          oacc[dt] = Elem<T>::mfma(as_vec8<T>(av), tr_pair<T>(t0 + 1024 * c + dt * kPanel, t1 + 1024 * c + dt * kPanel), oacc[dt]);
      }
      __builtin_amdgcn_s_setprio(0);
    }
    if (jt > 0) {      // the next tile is in LDS (the product just recorded may still be on its way), and this one has been read
      if (carry) vm_wait<1>(); else vm_wait<0>();
      lds_barrier();
    }
  }
  store_rows<T, DH, kLoadAligned>(p, tile, head, w_first, half, col, vb, oacc, prod);
}

// The products of fwd_dma_kernel rebuilt from q and k alone, bit for bit: 64 keys per barrier, K tiles straight into LDS one step ahead, and
// registers for five waves per SIMD, where the general kernel without V takes three, two barriers per 32 keys and LDS writes.  Bound by vector-ALU
// issue: 20 transcendentals at 16 cycles and 60 other instructions per 32 x 32 block beside 256 matrix cycles.  16 heads, 16384 tokens 102 -> 96 us.
template <typename T>
__global__ __launch_bounds__(kThreads, 4) void fwd_dma_carry_kernel(FwdParams p) {
  typedef typename Elem<T>::vec8 vec8;
  constexpr int DH = 128, kSteps = DH / 16, kPanel = 32 * 64, kMat = DH / 32 * kPanel, kBuf = 2 * kMat;      // bytes
  __shared__ __attribute__((aligned(16))) unsigned char lds_raw[2 * kBuf];
  lds_u8* const lds = (lds_u8*)lds_raw;
  const int lds_base = __builtin_amdgcn_readfirstlane((int)(uintptr_t)lds);
  int head, slot;
  xcd_head_tile(blockIdx.x, p.num_heads, &head, &slot);
  Tile tile;
  int64_t r0, r1;
  if (!forward_tile(p, slot, 0, kBlockQ, &tile, &r0, &r1)) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, col = lane & 31;
  const int L = tile.seq_len, q0 = tile.origin, ac = p.attend_current;
  const T* qb = (const T*)p.q.ptr + tile.seq_id * p.q.sb + head * p.q.sh + (int64_t)tile.seq_start * p.q.st;
  const T* kb = (const T*)p.k.ptr + tile.seq_id * p.k.sb + head * p.k.sh + (int64_t)tile.seq_start * p.k.st;
  const int last_key = min(q0 + kBlockQ, L) - 2 + ac;        // last key any row of this tile can see
  const int n_kt = last_key < 0 ? 0 : last_key / 32 + 1, n_pt = (n_kt + 1) >> 1;
  if (n_pt == 0) return;
  const int w_first = q0 + wave * 32, w_last = w_first + 31, qi = w_first + col;

  // Keys 64 pt .. into buffer pt & 1: a wave brings one panel of either half.  Row m is key mfma_row_to_key32(m): the MFMA's output row.
  const int k_st = (int)(p.k.st * 2);
  const u32x4 desc = buffer_desc(kb, (L - 1) * k_st + 2 * DH);
  const int voff = mfma_row_to_key32(lane >> 2) * k_st + 64 * wave + (((lane & 3) ^ ((lane >> 4) & 3)) << 4);
  auto request = [&](int pt) {
    const int dst = lds_base + (pt & 1) * kBuf + wave * kPanel;
#pragma unroll
    for (int i = 0; i < 2; i++) dma16x2<1024>(dst + i * kMat, voff, desc, (64 * pt + 32 * i) * k_st, (64 * pt + 32 * i + 8) * k_st);
  };
  request(n_pt - 1);
  vec8 qf[kSteps];
  load_operand<T, kLoadAligned>(qf, make_row_source<T, kLoadAligned>(qb, p.q.st, L, DH), qi, half);
  float prod = 1.f;    // prod over the keys already swept of (1 - sigma): both half-waves hold the same value
  const int n_qt = (L + kBlockQ - 1) / kBlockQ;
  // (A last pair whose upper half no row sees: its product is the empty one, which the backward kernels that sweep 64 keys read.)
  const uint32_t lrow = wave * 32 + col;
  const int top = 2 * n_pt - 1;
  float* row = p.carry + (int64_t)head * p.carry_head_stride + tile.carry_base + carry_offset(top, n_qt) + (q0 - kBlockQ * (top >> 2));
  const int row_a = col * 64 + ((half ^ ((col >> 2) & 3)) << 4);      // odd steps: ^ 32
  vm_wait<0>();
  lds_barrier();
  for (int pt = n_pt - 1; pt >= 0; --pt) {
    if (pt > 0) request(pt - 1);
#pragma unroll
    for (int i = 1; i >= 0; --i) {
      const int jt = 2 * pt + i, j0 = 32 * jt;
      if (half == 0) row[lrow] = prod;
      row -= carry_step(jt - 1, n_qt);
      if (j0 > w_last - 1 + ac) continue;                     // nothing visible to this wave yet
      const bool diagonal = (j0 + 31) > (w_first - 1 + ac);
      __builtin_amdgcn_s_setprio(3);
      f32x16 s[1];
#pragma unroll
      for (int r = 0; r < 16; r++) s[0][r] = 0.f;
      lds_u8* k0 = lds + (pt & 1) * kBuf + i * kMat + row_a;
      lds_u8* k1 = lds + (pt & 1) * kBuf + i * kMat + (row_a ^ 32);
      auto k_op = [&](int kk) { return lds_load<vec8>(((kk & 1) ? k1 : k0) + (kk >> 1) * kPanel); };
      vec8 a[4];
#pragma unroll
      for (int kk = 0; kk < 4; kk++) a[kk] = k_op(kk);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < kSteps; kk++) {
        s[0] = Elem<T>::mfma(a[kk & 3], qf[kk], s[0]);
        if (kk + 4 < kSteps) a[kk & 3] = k_op(kk + 4);
        __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_s_setprio(0);
      Weights<16> w;
      const int lim = qi + ac - j0 - 16 * half;               // key R is visible iff R < lim
      if (diagonal) w.template front<true>(s, p.scale_log2, lim); else w.template front<false>(s, p.scale_log2, lim);
      prod = (prod * other_half(w.run, half)) * w.run;
    }
    if (pt > 0) {      // the next keys are in LDS (the two products just recorded may still be on their way), and these have been read
      vm_wait<2>();
      lds_barrier();
    }
  }
}

template <typename T, bool kCarryOnly>
static hipError_t launch_fwd_t(const FwdParams& p, int max_tiles, hipStream_t stream) {
  const dim3 grid((unsigned)(max_tiles * p.num_heads + p.sched.service)), block(kThreads);
  if (p.load == kLoadAligned) {
    if (p.head_dim == 128 && !kCarryOnly) hipLaunchKernelGGL((fwd_dma_kernel<T>), grid, block, 0, stream, p);
    else if (p.head_dim == 128) hipLaunchKernelGGL((fwd_dma_carry_kernel<T>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((fwd_kernel<T, 64, kLoadAligned, 64, 2, kCarryOnly>), grid, block, 0, stream, p);
  } else if (p.load == kLoadPadded) {
    if (p.head_dim > 64) hipLaunchKernelGGL((fwd_kernel<T, 128, kLoadPadded, 32, 3, kCarryOnly>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((fwd_kernel<T, 64, kLoadPadded, 64, 2, kCarryOnly>), grid, block, 0, stream, p);
  } else {
    if (p.head_dim > 64) hipLaunchKernelGGL((fwd_kernel<T, 128, kLoadScalar, 64, 2, kCarryOnly>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((fwd_kernel<T, 64, kLoadScalar, 64, 2, kCarryOnly>), grid, block, 0, stream, p);
  }
  return hipGetLastError();
}

hipError_t launch_fwd(const FwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream) {
  return dtype_is_f16 ? launch_fwd_t<_Float16, false>(p, max_tiles, stream)
                      : launch_fwd_t<__bf16, false>(p, max_tiles, stream);
}

// The products the backward starts from, rebuilt from q and k alone (p.carry must be set; o, rem, row_stat, v unused).
hipError_t launch_fwd_carry_only(const FwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream) {
  return dtype_is_f16 ? launch_fwd_t<_Float16, true>(p, max_tiles, stream)
                      : launch_fwd_t<__bf16, true>(p, max_tiles, stream);
}

}  // namespace sba
