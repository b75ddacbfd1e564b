// Backward of sequences of up to 64 tokens: dq, dk and dv of one (head, sequence) by one workgroup of two waves, from one evaluation of S, dP and the
// tile math.
//
// What bounds such sequences is memory: 32 tokens x 128 are 57 KB of tensors and 3 x 40 matrix instructions.  The kernels of longer ones read Q, K,
// V and dO twice (dQ, then dK/dV) and give a workgroup of four or eight waves to rows that fill one or two.  Here wave b has rows 32 b .. of the
// sequence and then its keys 32 b ..: K and V go to LDS, Q and dO stay in registers; P and dZ of the (up to three) 32 x 32 blocks are left in LDS
// while dQ is summed; then dO and Q take the places of V and K, and each wave contracts its keys' columns of P and dZ over the rows.  Two barriers,
// nothing read twice, no sums between workgroups.  52 KB of LDS (head_dim 64: 32): three (five) workgroups per compute unit cover each other's loads.
// The forward's products (`carry`) are read as by the other kernels.  32 heads x 128, 2048 sequences of 1 to 64 tokens: 919 us, 3.8e9 bytes at 4.1 TB/s
// (dQ and dK/dV kernels 2138); head_dim 64 468 (1060).  (When it runs stands with tiny_of in sba_api.hip.)
#include "sba_device.hpp"
#include "sba_host.hpp"
#include "sba_params.hpp"

#include <type_traits>

namespace sba {

constexpr int kTinyThreads = 128;
constexpr int kTinyPzStride = 36;      // elements per row of a block of P or dZ in LDS

// An accumulator tile (row 8 * (r / 4) + 4 * half + r % 4, column 32 * dt + col) to memory; `scratch`: 32 x kTinyPzStride elements of the wave's own.
template <typename T, int DH, int kLoad>
__device__ __forceinline__ void store_tiny(const RowSink<T>& sink, const f32x16 (&acc)[DH / 32], float scale, int row0, int half, int col, int lane, int D, T* scratch) {
#pragma unroll
  for (int dt = 0; dt < DH / 32; dt++) {
    if (kLoad == kLoadAligned) store_acc_tile_wide<T, kTinyPzStride>(sink, acc[dt], scale, row0, 32 * dt, half, col, lane, scratch);
    else store_acc_tile<T>(sink, acc[dt], scale, row0, 32 * dt, half, col, D);
  }
}

template <typename T, int DH, int kLoad>
__global__ __launch_bounds__(kTinyThreads, 2) void bwd_tiny_kernel(BwdParams p) {
  constexpr int kSteps = DH / 16, kDTiles = DH / 32, kStride = lds_stride<DH>(), kBlock = 32 * kTinyPzStride;
  typedef typename Elem<T>::vec8 vec8;
  __shared__ __attribute__((aligned(16))) T kq_lds[64 * kStride];           // K, then Q
  __shared__ __attribute__((aligned(16))) T vo_lds[64 * kStride];           // V, then dO
  __shared__ __attribute__((aligned(16))) T pz_lds[3][2][kBlock];           // {P, dZ} of the blocks (rows, keys) 00, 10, 11: [row][key]
  int head, slot;
  xcd_head_tile(blockIdx.x, p.num_heads, &head, &slot);
  if (slot >= p.counts[kCountQ]) {
    int64_t r0, r1;
    if (p.tiny == kTinyAll && uncovered_rows(p.counts, slot, p.total_tokens, 0, kBlockQ, &r0, &r1)) {      // rows of no sequence: zero gradients
      zero_rows<T>(p.dq, head, r0, r1, p.head_dim);
      zero_rows<T>(p.dk, head, r0, r1, p.head_dim);
      zero_rows<T>(p.dv, head, r0, r1, p.head_dim);
    }
    return;
  }
  const Tile tile = p.q_tiles[slot];
  const int L = tile.seq_len;
  if (L > kTinyRows) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, col = lane & 31;
  const int ac = p.attend_current, D = kLoad == kLoadPadded ? p.head_dim : DH;
  const int64_t tok0 = tile.seq_start;
  const int first = 32 * wave, qi = first + col;
  const bool here = first < L;                                              // whether this wave has rows (and keys)
  const RowSource<T> qsrc = make_row_source<T, kLoad>((const T*)p.q.ptr + tile.seq_id * p.q.sb + head * p.q.sh + tok0 * p.q.st, p.q.st, L, D),
                     ksrc = make_row_source<T, kLoad>((const T*)p.k.ptr + tile.seq_id * p.k.sb + head * p.k.sh + tok0 * p.k.st, p.k.st, L, D),
                     vsrc = make_row_source<T, kLoad>((const T*)p.v.ptr + tile.seq_id * p.v.sb + head * p.v.sh + tok0 * p.v.st, p.v.st, L, D),
                     dosrc = make_row_source<T, kLoad>((const T*)p.d_o.ptr + tile.seq_id * p.d_o.sb + head * p.d_o.sh + tok0 * p.d_o.st, p.d_o.st, L, D);
  T* const kq_mine = kq_lds + first * kStride;
  T* const vo_mine = vo_lds + first * kStride;
  vec8 qf[kSteps], dof[kSteps];
  float drem = 0.f, prod[2] = {1.f, 1.f};      // prod: above key block 0 and above key block 1
  const int last_key = min(first + 32, L) - 2 + ac;                         // last key that a row of this wave sees
  if (here) {
    TileCopy<T, DH, 32, kLoad, 64> ck, cv;
    ck.load(ksrc, first);
    cv.load(vsrc, first);
    load_operand<T, kLoad>(qf, qsrc, qi, half);
    load_operand<T, kLoad>(dof, dosrc, qi, half);
    const float* carry = p.carry + (int64_t)head * p.carry_head_stride + tile.carry_base + qi;
    if (last_key >= 0) prod[0] = carry[0];
    if (last_key >= 32) prod[1] = carry[kBlockQ];
    if (qi < L && p.d_rem.ptr) drem = (float)((const T*)p.d_rem.ptr)[tile.seq_id * p.d_rem.sb + head * p.d_rem.sh + (tok0 + qi) * p.d_rem.st];
    ck.store(kq_mine);
    cv.store(vo_mine);
  }
  __syncthreads();
  f32x16 acc[kDTiles];
#pragma unroll
  for (int dt = 0; dt < kDTiles; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[dt][r] = 0.f;
  if (here) {
    if (p.add_rem) {      // the forward wrote o + rem * v: the gradient reaching rem is d_rem + d_o . v_i
      float dot = 0.f;
#pragma unroll
      for (int kk = 0; kk < kSteps; kk++) {
        const vec8 vf = lds_row8<T>(vo_mine, kStride, col, 16 * kk + 8 * half);
#pragma unroll
        for (int t = 0; t < 8; t++) dot = fmaf((float)dof[kk][t], (float)vf[t], dot);
      }
      drem += dot + other_half(dot, half);
    }
    const int krow = mfma_row_to_key32(col);
    float prefix = 0.f;
    for (int u = 0; u <= wave; u++) {
      T* const p_out = pz_lds[wave + u][0] + col * kTinyPzStride + 16 * half;
      uint32_t pk[8], dzk[8];
      if (32 * u <= last_key) {
        f32x16 s[1], dp[1];
#pragma unroll
        for (int r = 0; r < 16; r++) { s[0][r] = 0.f; dp[0][r] = 0.f; }
#pragma unroll
        for (int kk = 0; kk < kSteps; kk++) s[0] = Elem<T>::mfma(lds_row8<T>(kq_lds + 32 * u * kStride, kStride, krow, 16 * kk + 8 * half), qf[kk], s[0]);
#pragma unroll
        for (int kk = 0; kk < kSteps; kk++) dp[0] = Elem<T>::mfma(lds_row8<T>(vo_lds + 32 * u * kStride, kStride, krow, 16 * kk + 8 * half), dof[kk], dp[0]);
        // (dZ in the form, and so with the bits, of the kernels that form dQ alone; P beside it)
        BwdMath<16> m;
        const int lim = qi < L ? qi + ac - 32 * u - 16 * half : 0;
        if (u == wave || first + 31 >= L) bwd_math_front<1, true, false>(m, s, dp, p.scale_log2, lim, half, drem, u ? prod[1] : prod[0]);
        else bwd_math_front<1, false, false>(m, s, dp, p.scale_log2, lim, half, drem, u ? prod[1] : prod[0]);
        float above = m.seed;
#pragma unroll
        for (int i = 7; i >= 0; --i) {
          const float a1 = m.beta[2 * i + 1] * above, between = m.pe[2 * i + 1] * m.seed;
          pk[i] = pack2<T>(m.beta[2 * i] * between, a1);
          above = m.pe[2 * i] * m.seed;
        }
        uint32_t none[8];
        bwd_math_back<T, 16, false>(m, prefix + (half ? m.oth_g : 0.f), none, dzk);
        prefix += m.tot + m.oth_g;
#pragma unroll
        for (int c = 0; c < 2; c++) {
          const vec8 a = as_vec8<T>(u32x4{dzk[4 * c], dzk[4 * c + 1], dzk[4 * c + 2], dzk[4 * c + 3]});
#pragma unroll
          for (int dt = 0; dt < kDTiles; dt++) acc[dt] = Elem<T>::mfma(a, lds_col8<T>(kq_lds + 32 * u * kStride, kStride, 16 * half + 8 * c, 32 * dt, lane), acc[dt]);
        }
      } else {
#pragma unroll
        for (int i = 0; i < 8; i++) pk[i] = dzk[i] = 0u;
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {      // (rows of 72 bytes)
        *reinterpret_cast<u32x2*>(p_out + 4 * i) = u32x2{pk[2 * i], pk[2 * i + 1]};
        *reinterpret_cast<u32x2*>(p_out + kBlock + 4 * i) = u32x2{dzk[2 * i], dzk[2 * i + 1]};
      }
    }
  }
  __syncthreads();      // K and V have been read
  if (here) {
    const RowSink<T> sink = make_row_sink<T>((T*)p.dq.ptr + tile.seq_id * p.dq.sb + head * p.dq.sh + tok0 * p.dq.st, p.dq.st, L, D);
    store_tiny<T, DH, kLoad>(sink, acc, p.logit_scale, first, half, col, lane, D, kq_mine);
#pragma unroll
    for (int kk = 0; kk < kSteps; kk++) {
      *reinterpret_cast<vec8*>(kq_mine + col * kStride + 16 * kk + 8 * half) = qf[kk];
      *reinterpret_cast<vec8*>(vo_mine + col * kStride + 16 * kk + 8 * half) = dof[kk];
    }
  }
  __syncthreads();
  if (!here) return;
  const int blocks = L > 32 ? 2 : 1;
  T* const scratch = pz_lds[2 * wave][0];      // of the block on the diagonal, which no other wave reads
  // dV, then dK, of this wave's keys.
#pragma unroll 1
  for (int out = 0; out < 2; out++) {
#pragma unroll
    for (int dt = 0; dt < kDTiles; dt++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[dt][r] = 0.f;
    const T* const rows = out ? kq_lds : vo_lds;
    for (int b = wave; b < blocks; b++) {
      const T* const w = pz_lds[b + wave][out];
#pragma unroll
      for (int c = 0; c < 2; c++) {
        const int row0 = 16 * c + 8 * half;
        const vec8 a = lds_col8<T>(w, kTinyPzStride, row0, 0, lane);
#pragma unroll
        for (int dt = 0; dt < kDTiles; dt++) acc[dt] = Elem<T>::mfma(a, lds_col8<T>(rows + 32 * b * kStride, kStride, row0, 32 * dt, lane), acc[dt]);
      }
    }
    if (!out && p.add_rem) {      // the forward wrote o + rem * v: dv_i gains rem_i * d_o_i
      const float rem = fast_exp2(p.row_stat[tile.seq_id * p.stat_sb + head * p.stat_sh + tok0 + min(qi, L - 1)]);
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int row = 8 * (r >> 2) + 4 * half + (r & 3);
        const float rem_row = __shfl(rem, row);
#pragma unroll
        for (int dt = 0; dt < kDTiles; dt++) acc[dt][r] = fmaf(rem_row, (float)vo_mine[row * kStride + 32 * dt + col], acc[dt][r]);
      }
    }
    // (the scratch lies over P of the block on the diagonal, which has been read)
    const TensorRef& t = out ? p.dk : p.dv;
    const RowSink<T> sink = make_row_sink<T>((T*)t.ptr + tile.seq_id * t.sb + head * t.sh + tok0 * t.st, t.st, L, D);
    store_tiny<T, DH, kLoad>(sink, acc, out ? p.logit_scale : 1.f, first, half, col, lane, D, scratch);
  }
}

hipError_t launch_bwd_tiny(const BwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream) {
  auto launch = [&](auto t, auto dh, auto load) {
    hipLaunchKernelGGL((bwd_tiny_kernel<decltype(t), decltype(dh)::value, decltype(load)::value>), dim3((unsigned)(max_tiles * p.num_heads)), dim3(kTinyThreads), 0,
                       stream, p);
    return hipGetLastError();
  };
  auto by_load = [&](auto t, auto dh) {
    return p.load == kLoadAligned ? launch(t, dh, std::integral_constant<int, kLoadAligned>()) : launch(t, dh, std::integral_constant<int, kLoadPadded>());
  };
  auto by_dim = [&](auto t) { return p.head_dim > 64 ? by_load(t, std::integral_constant<int, 128>()) : by_load(t, std::integral_constant<int, 64>()); };
  return dtype_is_f16 ? by_dim(_Float16()) : by_dim((__bf16)0.f);
}

}  // namespace sba
