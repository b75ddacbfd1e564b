// Backward on row tiles: dq, dk and dv from ONE evaluation of S, dP and the tile math per visible (query, key) pair.
//
// One workgroup = 8 waves = one tile of 256 query rows of one (head, sequence), 32 rows per wave (lane l owns query l%32), which
// sweeps the keys UPWARDS from key 0 to its diagonal in blocks of 32.  C, the prefix sum of g along a row, therefore stays in a
// register, and dQ is accumulated in registers as in the dQ kernel (sba_bwd_dq.hip).  What crosses rows is dK and dV: every wave
// leaves its P and dZ of the block in LDS, and each of the 8 waves contracts one 32 x 32 piece of {dV, dK} over the 256 rows, dO or Q
// as stationary operands in registers.  The piece is added to what the row tile ABOVE left of it in memory and left for the row
// tile below; the tile that holds the keys' own rows converts and stores the result.  So the row tiles of a (head, sequence) form
// a chain: the last one (whose sweep is longest) starts, and a tile follows the one above it a block or two behind.  Each sum is
// formed in one fixed order: the same bits every time, no atomics (the reference adds dK and dV tiles behind a spin lock:
// stickbreaking_attention/sb_varlen/sb_varlen_bwd.py:11-53).
//
// Hand-over.  A wave issues its stores, waits for them (vmcnt) and then stores the number of key blocks that are complete into a flag of
// its own; the same wave of the tile below reads flag and partial results with sc1 (served by the L2, never by the vector L1).  All
// tiles of a (head, sequence) run on one XCD, i.e. on one L2: (head, sequence) belongs to one of 8 queues (row_queue), a workgroup takes
// tiles from queue blockIdx % 8 (workgroups are dealt to the XCDs in turn), and every workgroup checks its XCC id against the first
// of its queue: one that is elsewhere leaves.  Progress: the tiles of chains are taken in list order, a tile waits only for one that was taken before
// it, so every wait ends; the waits are bounded all the same.  A tile whose wait ran out passes on NaN and a count that says so
// (kChainBroken; data alone would not do, the tile above may still overwrite it), and stores NaN: no wrong number leaves the kernel.
//
// What bounds it: per 32 x 32 block and wave 40 MFMAs (1280 cycles), 320 vector-ALU instructions and 48 KB of LDS reads, two waves per
// SIMD.  The waves of a SIMD (w and w + 4) are kept out of step: one contracts the block of the step before at the start of a
// step, the other at its end (32 heads x 8 x 4096: 4970 -> 4660 us per training pass).  32 heads x 8 x 4096 x 128, one pass of
// the backward: 4180 us with key tiles (sba_bwd_chain.hip), 3330 us here; 32768 tokens in 25 sequences of up to 4096, 32 heads: 2650 and
// 2000.  A step takes 5800 cycles.  Either pipe of a SIMD is busy 78 % of the time (69 % on the 25 sequences), both 7 to 9 %; waves wait 35 % (39 %) of
// theirs.  Without the hand-over it would take 3130 of 3300, without the tile math as well 2590: at 2.1 GHz, the clock that the power limit
// leaves, and 2.0 for the products alone.  256 rows per tile, because the hand-over costs 8 bytes per pair / (rows / 256).  The next tile of a workgroup
// costs 27000 cycles (17.8 tiles of 34 steps each on the 25 sequences): 11000 to 17000 for its Q and dO, behind the other workgroups' traffic, 3000
// for dQ, 2300 for its place in the list.
//
// head_dim 64: half the products per pair and the same element-wise work (320 vector-ALU instructions against 20 MFMAs per block and
// wave); vector ALU busy 51 %, either pipe 69 %, and waves wait 40 % of their time: two waves per SIMD that meet at two barriers per step
// bound it.  A key block has four pieces of {dV, dK}, so a step is two blocks and a wave contracts a piece of one of
// them; LDS holds four blocks, Q stays in registers.  (Steps of one block, contracted by every second wave in turn: the wave whose
// turn it is arrives last at every barrier: 12 heads, 16384 tokens in 10 sequences of up to 3523, 474 us instead of 434.)  Training passes,
// us, two kernels and here: 484 and 434; 16 heads x 4 x 4096 946 and 763; 8 heads x 8 x 1024 142 and 108.
#include "sba_device.hpp"
#include "sba_dma.hpp"
#include "sba_host.hpp"
#include "sba_params.hpp"

#include <atomic>
#include <type_traits>

namespace sba {

constexpr int kRowTile = kRowTileRows;      // query rows per workgroup
constexpr int kRowWaves = 8, kRowThreads = 64 * kRowWaves;
constexpr int kRowKeys = 32;                // keys per step

template <int DH>
struct RowLds {
  static constexpr int kBufs = DH == 128 ? 2 : 4;      // of the key blocks' buffers: two steps' worth
  static constexpr int kExch = 0;                      // {P, dZ} of a block: [row][32 keys], 16 KB each
  static constexpr int kExchBuf = 32768, kExchMat = 16384;
  static constexpr int kQ = 65536;                     // Q of the tile: panels of [row][32 columns] (head_dim 64: until it is in registers)
  static constexpr int kPanels = DH / 32, kPanel = kRowTile * 64;
  static constexpr int kKv = 131072;                   // {K, V} of a block: panels of [key][32 columns] each
  static constexpr int kKvPanel = kRowKeys * 64, kKvMat = kPanels * kKvPanel, kKvBuf = 2 * kKvMat;
  static constexpr int kBytes = kKv + kBufs * kKvBuf;
};

__device__ __forceinline__ void lds_put(lds_u8* p, u32x4 v) { *reinterpret_cast<__attribute__((address_space(3))) u32x4*>(p) = v; }
// x ^ kBit, computed where it is used: kept over the loop it would cost a register the loop does not have.
template <int kBit>
__device__ __forceinline__ int flip(int x) {
  int r;
  asm volatile("v_xor_b32 %0, %1, %2" : "=v"(r) : "n"(kBit), "v"(x));
  return r;
}

// The tile math of 32 rows x 32 keys (bwd_math_front / bwd_math_back) in two parts, so that dP need not be there for the first:
// P, which leaves for LDS at once, and sigma and the products below each key for the second.
template <typename T>
struct RowMath {
  float beta[16], pe[16], seed;
  // s: base-2 logits, -inf where hidden.
  __device__ __forceinline__ void weights(const f32x16& s, int half, float prod_in, lds_u8* p_out) {
    float run = 1.f;
#pragma unroll
    for (int R = 15; R >= 0; --R) {
      const float omb = fast_rcp(1.f + fast_exp2(s[R]));
      beta[R] = 1.f - omb;
      run *= omb;
      pe[R] = run;
    }
    const float oth = other_half(run, half);
    seed = half ? prod_in : prod_in * oth;
    float above = seed;
#pragma unroll
    for (int i = 1; i >= 0; --i) {
      float a[8];
#pragma unroll
      for (int r = 7; r >= 0; --r) {
        const int R = 8 * i + r;
        a[r] = beta[R] * above;
        above = pe[R] * seed;
        pe[R] = above;
      }
      lds_put(i ? (lds_u8*)(uintptr_t)((int)(uintptr_t)p_out ^ 16) : p_out, u32x4{pack2<T>(a[0], a[1]), pack2<T>(a[2], a[3]), pack2<T>(a[4], a[5]), pack2<T>(a[6], a[7])});
    }
  }
  __device__ __forceinline__ void gradients(const f32x16& dp, int half, float drem, float& prefix, u32x4 (&dz)[2]) {
    float u[16], D = drem;
#pragma unroll
    for (int R = 0; R < 16; R++) {
      u[R] = dp[R] - D;
      D = fmaf(beta[R], u[R], D);
    }
    const float tot = (D - drem) * seed, oth_g = other_half(tot, half);
    const float below = prefix + (half ? oth_g : 0.f);
    prefix += tot + oth_g;
#pragma unroll
    for (int i = 0; i < 8; i++)
      dz[i >> 2][i & 3] = pack2<T>(beta[2 * i] * fmaf(pe[2 * i], u[2 * i], -below), beta[2 * i + 1] * fmaf(pe[2 * i + 1], u[2 * i + 1], -below));
  }
};

// The lane's number, computed where it is used (see flip).
__device__ __forceinline__ int this_lane() {
  int r;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(r));
  return r;
}

// acc += rem * d_o for the 32 rows that the operands wf[2 kk] and wf[2 kk + 1] hold; rem: of row `col`.  An operand's lane holds rows
// 8 half + t, the accumulator's 8 (r >> 2) + 4 half + (r & 3): the half-waves swap every second pair of pairs.  (d_o read again from
// memory, element by element in the accumulator's layout: 1101 us instead of 927 for a training pass of 16 heads, 16384 tokens in f16.)
template <typename T>
__device__ __forceinline__ void add_rem_rows(f32x16& acc, const typename Elem<T>::vec8 (&wf)[16], int kk, float rem, int half) {
  typedef __attribute__((ext_vector_type(2))) T pair;
  u32x4 x[2] = {};
#pragma unroll
  for (int k = 0; k < 8; k++)
    if (k == kk) { x[0] = __builtin_bit_cast(u32x4, wf[2 * k]); x[1] = __builtin_bit_cast(u32x4, wf[2 * k + 1]); }
#pragma unroll
  for (int c = 0; c < 2; c++)
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const auto y = __builtin_amdgcn_permlane32_swap(x[c][i], x[c][i + 2], false, false);
#pragma unroll
      for (int g = 0; g < 2; g++) {
        const uint32_t bits = y[g];
        const pair d = __builtin_bit_cast(pair, bits);
#pragma unroll
        for (int e = 0; e < 2; e++) {
          const int r = 8 * c + 4 * g + 2 * i + e;
          acc[r] = fmaf(__shfl(rem, 8 * (r >> 2) + 4 * half + (r & 3)), (float)d[e], acc[r]);
        }
      }
    }
}

// The kernel's arguments, read where they are needed and not kept in scalar registers, which the loop is short of.
typedef const __attribute__((address_space(4))) BwdParams Args;
__device__ __forceinline__ Args* kernel_args() {
  Args* args = (Args*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(args));
  return args;
}

// Until the tile above has passed on more than t key blocks: how many it has.
__device__ __forceinline__ int wait_for(const int32_t* pred, int t, int lane) {
  Args* args = kernel_args();
  const int polls = args->wait_polls;
  int v = 0;
#pragma unroll 1
  for (int spins = 0; spins < polls; spins++) {
    asm volatile("s_nop 4\n\tglobal_load_dword %0, %1, %2 sc1\n\ts_waitcnt vmcnt(0)" : "=v"(v) : "v"(0), "s"(pred) : "memory");
    v = __builtin_amdgcn_readfirstlane(v);
    if (v > t) return v;
    __builtin_amdgcn_s_sleep(1);
  }
  if (lane == 0) atomicMax(args->status, kSchedChainTimeout);
  return kChainBroken;      // no later wait of this tile
}

template <typename T, int DH, bool kAddRem>
__global__ __launch_bounds__(kRowThreads, 2) void bwd_row_kernel(BwdParams p) {
  constexpr int kSteps = DH / 16, kDTiles = DH / 32;
  constexpr bool kWide = DH == 128;        // a step is one key block, of which every wave contracts a piece; else two, of which it contracts one
  constexpr int kPieces = DH / 16;         // 32 x 32 pieces of dV and dK per key block
  typedef RowLds<DH> Lds;
  typedef typename Elem<T>::vec8 vec8;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  lds_u8* const lds = (lds_u8*)lds_raw;
  const int lds_base = __builtin_amdgcn_readfirstlane((int)(uintptr_t)lds);

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, col = lane & 31;
  const int ac = p.attend_current, H = p.num_heads;
  const int queue = blockIdx.x & 7;
  int32_t* const cursor = (int32_t*)p.chain_c + queue;

  if (threadIdx.x == 0) {
    const int xcc = (int)(__builtin_amdgcn_s_getreg((20) | (0 << 6) | ((4 - 1) << 11)) & 15) + 1;     // HW_REG_XCC_ID
    const int old = atomicCAS(p.chain_head_xcc + queue, 0, xcc);
    *reinterpret_cast<int*>(lds_raw) = old != 0 && old != xcc;
  }
  // Rows of the packed token axis that belong to no sequence: zero gradients.
  {
    const int64_t covered = p.counts[kCountCovered];
    if (covered < p.total_tokens) {
      const int parts = ((int)gridDim.x + H - 1) / H;
      const int64_t n = p.total_tokens - covered, per = (n + parts - 1) / parts;
      for (int i = blockIdx.x; i < parts * H; i += gridDim.x) {
        const int64_t a = covered + per * (i / H), b = a + per < p.total_tokens ? a + per : p.total_tokens;
        if (a < b) {
          zero_rows<T>(p.dq, i % H, a, b, DH);
          zero_rows<T>(p.dk, i % H, a, b, DH);
          zero_rows<T>(p.dv, i % H, a, b, DH);
        }
      }
    }
  }

  // A workgroup that is not on its queue's XCD leaves the tiles to those that are.
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(*reinterpret_cast<int*>(lds_raw))) return;
  __syncthreads();

  // Where a lane reads and writes in the panels: 64-byte rows whose 16-byte chunks are XORed with (row >> 2) & 3.
  const int sw = (col >> 2) & 3, s15 = lane & 15, g = (lane >> 4) & 1;
  const int row_a = col * 64 + ((half ^ sw) << 4);                                            // row reads; odd steps: ^ 32
  const int tr_chunk = 2 * g + ((s15 >> 1) & 1), tr_byte = 8 * (s15 & 1);
  const int tr_e = (8 * half + (s15 >> 2)) * 64 + ((tr_chunk ^ (2 * half)) << 4) + tr_byte;   // 4 rows down; the next 4: (^ 16) + 256
  const int tr_k = (4 * half + (s15 >> 2)) * 64 + ((tr_chunk ^ half) << 4) + tr_byte;         // ... in key order: (^ 32) + 512
  const int wr_a = (32 * wave + col) * 64 + (((2 * half) ^ sw) << 4);                         // 8 of this lane's keys; the others: ^ 16

  const bool out = kWide ? wave >= 4 : (wave & 2) != 0;      // which result this wave contracts: dK, else dV
  const int cp = kWide ? wave & 3 : wave & 1;           // ... and which 32 columns of it
  const int per_slot = (H + 7) >> 3;       // heads of a tile slot that a queue may hold
  // A queue has two lists: the tiles of chains, taken in order, and those that are their sequence's only one (no tile waits for them).  The latter
  // wait for memory most of their time, so some workgroups (apart_share in sba_params.hpp) begin with them while the others compute, and go over
  // to the other list when theirs is used up.  If none do, one list holds all.
  int chained, all;      // claims that chains have, and all (read again for each tile)
  auto read_lists = [&] {
    Args* args = kernel_args();
    const int32_t* counts = args->counts;
    const int n = counts[kCountK], slots = (args->num_heads + 7) >> 3, wgs = gridDim.x >> 3;
    const int begin_apart = apart_workgroups(wgs, counts[kCountApart]);
    all = __builtin_amdgcn_readfirstlane(n * slots);
    chained = begin_apart > 0 ? __builtin_amdgcn_readfirstlane(min(max(counts[kCountChained], 0), n) * slots) : all;
    return (int)(blockIdx.x >> 3) >= wgs - begin_apart;
  };
  bool apart = read_lists() && chained < all;

  for (;;) {
    if (threadIdx.x == 0) {
      int c = atomicAdd(cursor + (apart ? 8 : 0), 1) + (apart ? chained : 0);
      if (c >= (apart ? all : chained)) {      // that list is used up
        c = all;
        if (apart ? chained > 0 : chained < all) {
          c = atomicAdd(cursor + (apart ? 0 : 8), 1) + (apart ? 0 : chained);
          if (c >= (apart ? chained : all)) c = all;
        }
      }
      *reinterpret_cast<int*>(lds_raw) = c;
    }
    __syncthreads();
    const int claim = __builtin_amdgcn_readfirstlane(*reinterpret_cast<int*>(lds_raw));
    __syncthreads();
    apart = claim >= chained;
    if (claim >= all) break;
    const int place = claim / per_slot;
    Tile tile = p.k_tiles[place];
    const int first_slot = __builtin_amdgcn_readfirstlane(p.k_turns[place].first_slot), rank = __builtin_amdgcn_readfirstlane(p.k_turns[place].rank);
    const int L = __builtin_amdgcn_readfirstlane(tile.seq_len), seq_id = __builtin_amdgcn_readfirstlane(tile.seq_id);
    const int head = ((queue - row_queue(rank, H)) & 7) + 8 * (claim - place * per_slot);
    if (head >= H) continue;
    const int64_t tok0 = __builtin_amdgcn_readfirstlane(tile.seq_start);
    const int64_t carry_base = (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)tile.carry_base) |
                               (int64_t)__builtin_amdgcn_readfirstlane((int)(tile.carry_base >> 32)) << 32;
    // The list holds the tiles first to last; they are taken last to first.  They are laid from the sequence's end (a whole wave's 32 rows), so that
    // the one with fewer rows is the one that sweeps fewest keys: from row 0 on, a sequence of 300 rows took 8 + 10 key blocks, this way 2 + 10
    // (training passes, us: 32 heads, 32768 tokens in 25 sequences 2773 -> 2630, 12 heads x 64, 16384 tokens in 10 430 -> 412).
    const int nth = __builtin_amdgcn_readfirstlane(tile.origin) / kRowTile, slot = first_slot + nth;
    const int q_end = ((L + 31) & ~31) - nth * kRowTile, q0 = max(q_end - kRowTile, 0);
    const bool has_pred = nth > 0;
    const int n = q_end / kRowKeys;                                       // key blocks of this tile
    const int own = q0 / kRowKeys;                                        // the first of the tile's own rows' keys
    const int w_hi = (q_end - q0) / 32;                                   // waves with rows
    const bool has_rows = wave < w_hi;

    const T* qb = (const T*)p.q.ptr + seq_id * p.q.sb + head * p.q.sh + tok0 * p.q.st;
    const T* kb = (const T*)p.k.ptr + seq_id * p.k.sb + head * p.k.sh + tok0 * p.k.st;
    const T* vb = (const T*)p.v.ptr + seq_id * p.v.sb + head * p.v.sh + tok0 * p.v.st;
    const T* dob = (const T*)p.d_o.ptr + seq_id * p.d_o.sb + head * p.d_o.sh + tok0 * p.d_o.st;
    const int q_st = (int)(p.q.st * 2), do_st = (int)(p.d_o.st * 2);
    // K and V rows of step t's key blocks: a wave brings a panel of one of them (waves 0-3: K, 4-7: V; head_dim 64: of the first block, of
    // the second).
    const int kv_panel = kWide ? cp : wave & 1, kv_sub = kWide ? 0 : wave >> 2;
    const bool brings_v = kWide ? out : (wave & kDTiles) != 0;
    const int kv_st = (int)((brings_v ? p.v.st : p.k.st) * 2);
    const u32x4 kv_desc = buffer_desc(brings_v ? vb : kb, (L - 1) * kv_st + 2 * DH);
    const int kv_voff = mfma_row_to_key32(lane >> 2) * kv_st + kv_panel * 64 + (((lane & 3) ^ ((lane >> 4) & 3)) << 4);
    auto request_kv = [&](int t) {
      const int block = kWide ? t : 2 * t + kv_sub, soff = min(block, n - 1) * kRowKeys * kv_st;
      const int dst = kWide ? (t & 1) * Lds::kKvBuf + wave * 2048 : (block & 3) * Lds::kKvBuf + (wave & 3) * 2048;
      dma16x2<1024>(lds_base + Lds::kKv + dst, kv_voff, kv_desc, soff, soff + 8 * kv_st);
    };
    // Q and dO of the tile; dO into the exchange buffers until its operands are in registers.
    {
      const u32x4 q_desc = buffer_desc(qb, (L - 1) * q_st + 2 * DH), do_desc = buffer_desc(dob, (L - 1) * do_st + 2 * DH);
      const int chunk = ((lane & 3) ^ ((lane >> 4) & 3)) * 16;
      const int q_voff = (lane >> 2) * q_st + chunk, do_voff = (lane >> 2) * do_st + chunk;
#pragma unroll
      for (int i = 0; i < Lds::kPanels; i++) {      // panel i, rows 16 wave and 128 + 16 wave
        const int row = q0 + 16 * wave, dst = lds_base + wave * 1024 + i * Lds::kPanel;
        dma16x2<8192>(dst + Lds::kQ, q_voff, q_desc, row * q_st + 64 * i, (row + 128) * q_st + 64 * i);
        dma16x2<8192>(dst + Lds::kExch, do_voff, do_desc, row * do_st + 64 * i, (row + 128) * do_st + 64 * i);
      }
    }
    request_kv(0);
    const int w_first = q0 + 32 * wave, w_last = w_first + 31, qi = w_first + col;
    const bool row_ok = qi < L;
    float drem = 0.f;
    if (row_ok && p.d_rem.ptr) drem = (float)((const T*)p.d_rem.ptr)[seq_id * p.d_rem.sb + head * p.d_rem.sh + (tok0 + qi) * p.d_rem.st];
    // The forward's product above key block u for this lane's row (kept within what was recorded).
    const int n_qt = (L + kBlockQ - 1) / kBlockQ;
    const int last_seen = min(w_last, L - 1) - 1 + ac;                    // last key a row of this wave sees
    const int u_last = has_rows && last_seen > 0 ? last_seen / kRowKeys : 0;
    const float* carry = p.carry + (int64_t)head * p.carry_head_stride + carry_base;
    const int row_c = min(qi, L - 1);
    auto product_at = [&](int t) {
      const int u = min(t, u_last);
      return carry + (carry_offset(u, n_qt) - kBlockQ * (u >> 2));
    };
    // What the row tiles of a (head, sequence) hand down: per key block and wave, the 32 x 32 partial result.  (Sequences of more than one
    // tile have the first slots, each with 8 key blocks per tile.)
    const int64_t first_block = p.chain_by_slot ? (int64_t)first_slot * (kRowTile / kRowKeys) : tok0 * 9 / 256;
    float* part = p.chain_dq + ((int64_t)head * p.chain_rows + first_block) * (kPieces * 1024) + (wave & (kPieces - 1)) * 1024;
    int32_t* flag = p.chain_flags + ((int64_t)head * p.chain_tile_cap + slot) * 8 + wave;
    const int32_t* pred = has_pred ? flag - 8 : flag;
    const int lane16 = lane * 16;

    vm_wait<0>();
    __syncthreads();
    vec8 dof[kSteps], wf[16], qf[kWide ? 1 : kSteps];
    if constexpr (!kWide) {      // (head_dim 128: read from LDS in every step)
      lds_u8* rows = lds + Lds::kQ + 32 * wave * 64;
#pragma unroll
      for (int kk = 0; kk < kSteps; kk++) qf[kk] = lds_load<vec8>(rows + ((kk & 1) ? row_a ^ 32 : row_a) + (kk >> 1) * Lds::kPanel);
    }
    {
      lds_u8* rows = lds + Lds::kExch + 32 * wave * 64;
#pragma unroll
      for (int kk = 0; kk < kSteps; kk++) dof[kk] = lds_load<vec8>(rows + ((kk & 1) ? row_a ^ 32 : row_a) + (kk >> 1) * Lds::kPanel);
      lds_u8* cols = lds + (out ? Lds::kQ : Lds::kExch) + cp * Lds::kPanel;
#pragma unroll
      for (int c = 0; c < 16; c++) wf[c] = tr_pair<T>(cols + tr_e + 1024 * c, cols + (tr_e ^ 16) + 256 + 1024 * c);
    }
    if (kAddRem) {      // the forward wrote o + rem * v: the gradient reaching rem is d_rem + d_o . v_i
      float dot = 0.f;
      const RowSource<T> vsrc = make_row_source<T, kLoadAligned>(vb, p.v.st, L, DH);
#pragma unroll
      for (int kk = 0; kk < kSteps; kk++) {
        const vec8 vf = as_vec8<T>(__builtin_amdgcn_raw_buffer_load_b128(vsrc.rsrc, chunk_offset<T, kLoadAligned>(vsrc, qi, 16 * kk + 8 * half), 0, 0));
#pragma unroll
        for (int t = 0; t < 8; t++) dot = fmaf((float)dof[kk][t], (float)vf[t], dot);
      }
      drem += dot + other_half(dot, half);
    }
    f32x16 dqacc[kDTiles];
#pragma unroll
    for (int dt = 0; dt < kDTiles; dt++)
#pragma unroll
      for (int r = 0; r < 16; r++) dqacc[dt][r] = 0.f;
    float prefix = 0.f;

    const RowSink<T> sink = out ? make_row_sink<T>((T*)p.dk.ptr + seq_id * p.dk.sb + head * p.dk.sh + tok0 * p.dk.st, p.dk.st, L, DH)
                                : make_row_sink<T>((T*)p.dv.ptr + seq_id * p.dv.sb + head * p.dv.sh + tok0 * p.dv.st, p.dv.st, L, DH);
    float n_prod; float n_prod2;      // of the next step's key blocks
    int seen_count = 0;      // key blocks the tile above has passed on, as last read
    asm volatile("s_nop 4\n\tglobal_load_dword %0, %1, %2" : "=v"(n_prod) : "v"(row_c * 4), "s"(product_at(0)) : "memory");
    if constexpr (!kWide) asm volatile("s_nop 4\n\tglobal_load_dword %0, %1, %2" : "=v"(n_prod2) : "v"(row_c * 4), "s"(product_at(1)) : "memory");
    if constexpr (kWide) asm volatile("s_waitcnt vmcnt(0)" : "+v"(n_prod)::"memory"); else asm volatile("s_waitcnt vmcnt(0)" : "+v"(n_prod), "+v"(n_prod2)::"memory");

    f32x4 c0 = {0.f, 0.f, 0.f, 0.f}, c1 = c0, c2 = c0, c3 = c0;      // what the tile above has passed on of the key block contracted next
    auto contract = [&](int tc) {
      const bool adds_rem = kAddRem && !out && tc >= own;      // dv_j gains rem_j * d_o_j
      f32x16 acc;
#pragma unroll
      for (int r = 0; r < 16; r++) acc[r] = 0.f;
      lds_u8* ex = lds + Lds::kExch + (tc & (Lds::kBufs - 1)) * Lds::kExchBuf + (out ? Lds::kExchMat : 0);
      lds_u8* e0 = ex + tr_e;
      lds_u8* e1 = ex + flip<16>(tr_e) + 256;
      const int w0 = max(0, tc - own);
      if (w0 == 0 && w_hi == kRowWaves) {
        vec8 a[4];
#pragma unroll
        for (int c = 0; c < 4; c++) a[c] = tr_pair<T>(e0 + 1024 * c, e1 + 1024 * c);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 16; c++) {
          acc = Elem<T>::mfma(a[c & 3], wf[c], acc);
          if (c + 4 < 16) a[c & 3] = tr_pair<T>(e0 + 1024 * (c + 4), e1 + 1024 * (c + 4));
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
#pragma unroll
        for (int kk = 0; kk < kRowWaves; kk++)
          if (kk >= w0 && kk < w_hi) {
#pragma unroll
            for (int c = 2 * kk; c < 2 * kk + 2; c++) acc = Elem<T>::mfma(tr_pair<T>(e0 + 1024 * c, e1 + 1024 * c), wf[c], acc);
          }
      }
      if (seen_count == kChainBroken) {      // (as a product: 16 registers set in a branch spilled 21 in the loop)
        vec8 nans;
#pragma unroll
        for (int i = 0; i < 8; i++) nans[i] = (T)NAN;
        acc = Elem<T>::mfma(nans, nans, acc);
      }
      asm volatile("s_waitcnt vmcnt(0)" : "+v"(c0), "+v"(c1), "+v"(c2), "+v"(c3)::"memory");
#pragma unroll
      for (int r = 0; r < 4; r++) { acc[r] += c0[r]; acc[4 + r] += c1[r]; acc[8 + r] += c2[r]; acc[12 + r] += c3[r]; }      // (zeros without a tile above)
      if (tc >= own) {
        if (adds_rem) {
          const int me = this_lane(), col = me & 31, half = me >> 5;
          add_rem_rows<T>(acc, wf, tc - own, fast_exp2(p.row_stat[seq_id * p.stat_sb + head * p.stat_sh + tok0 + min(kRowKeys * tc + col, L - 1)]), half);
        }
        store_acc_tile<T>(sink, acc, out ? p.logit_scale : 1.f, kRowKeys * tc, 32 * cp, half, col, DH);
      } else {
        const f32x4 d0 = __builtin_shufflevector(acc, acc, 0, 1, 2, 3), d1 = __builtin_shufflevector(acc, acc, 4, 5, 6, 7),
                    d2 = __builtin_shufflevector(acc, acc, 8, 9, 10, 11), d3 = __builtin_shufflevector(acc, acc, 12, 13, 14, 15);
        float* dst = part + (int64_t)tc * (kPieces * 1024);
        // (A store's data is read a wait state after it was issued, which the compiler does not keep for assembly either.)
        asm volatile("s_nop 4\n\tglobal_store_dwordx4 %0, %1, %5\n\tglobal_store_dwordx4 %0, %2, %5 offset:1024\n\t"
                     "global_store_dwordx4 %0, %3, %5 offset:2048\n\tglobal_store_dwordx4 %0, %4, %5 offset:3072\n\ts_nop 0"
                     ::"v"(lane16), "v"(d0), "v"(d1), "v"(d2), "v"(d3), "s"(dst) : "memory");
      }
    };
    const bool late = wave >= 4;      // (waves w and w + 4 share a SIMD)
    // Of a key block: P and dZ of this wave's rows, into LDS (`behind_weights` is done behind the first of them) ...
    auto front = [&](int j0, bool seen, lds_u8* kt, lds_u8* ex, float prod_in, u32x4 (&dz)[2], auto behind_weights) {
      if (seen) {
        f32x16 s, dp;
#pragma unroll
        for (int r = 0; r < 16; r++) { s[r] = 0.f; dp[r] = 0.f; }
        lds_u8* k0 = kt + row_a;
        lds_u8* k1 = kt + flip<32>(row_a);
        lds_u8* q0p = lds + Lds::kQ + 32 * wave * 64 + row_a;
        lds_u8* q1p = lds + Lds::kQ + 32 * wave * 64 + flip<32>(row_a);
        auto k_op = [&](int kk) { return lds_load<vec8>(((kk & 1) ? k1 : k0) + (kk >> 1) * Lds::kKvPanel); };
        auto v_op = [&](int kk) { return lds_load<vec8>(((kk & 1) ? k1 : k0) + Lds::kKvMat + (kk >> 1) * Lds::kKvPanel); };
        auto q_op = [&](int kk) {
          if constexpr (kWide) return lds_load<vec8>(((kk & 1) ? q1p : q0p) + (kk >> 1) * Lds::kPanel);
          else return qf[kk];
        };
        constexpr int kAhead = 3, kVAhead = 3;
        vec8 ka[kAhead], qa[kAhead], va[kVAhead];
#pragma unroll
        for (int kk = 0; kk < kAhead; kk++) { ka[kk] = k_op(kk); qa[kk] = q_op(kk); }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < kSteps; kk++) {
          s = Elem<T>::mfma(ka[kk % kAhead], qa[kk % kAhead], s);
          if (kk + kAhead < kSteps) { ka[kk % kAhead] = k_op(kk + kAhead); qa[kk % kAhead] = q_op(kk + kAhead); }
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] *= p.scale_log2;
        if (j0 + 31 > w_first - 1 + ac || w_last >= L) {      // hidden keys
          const int me = this_lane(), qi = w_first + (me & 31);
          const int lim = qi < L ? qi + ac - j0 - 16 * (me >> 5) : 0;
#pragma unroll
          for (int r = 0; r < 16; r++) s[r] = r < lim ? s[r] : -INFINITY;
        }
        RowMath<T> m;
        m.weights(s, half, prod_in, ex + wr_a);
        behind_weights();
#pragma unroll
        for (int kk = 0; kk < kVAhead; kk++) va[kk] = v_op(kk);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < kSteps; kk++) {
          dp = Elem<T>::mfma(va[kk % kVAhead], dof[kk], dp);
          if (kk + kVAhead < kSteps) va[kk % kVAhead] = v_op(kk + kVAhead);
          __builtin_amdgcn_sched_barrier(0);
        }
        m.gradients(dp, half, drem, prefix, dz);
      } else {
        behind_weights();
        vm_wait<0>();
        dz[0] = dz[1] = u32x4{0, 0, 0, 0};
        lds_put(ex + wr_a, dz[0]);
        lds_put(ex + (wr_a ^ 16), dz[0]);
      }
      lds_put(ex + Lds::kExchMat + wr_a, dz[0]);
      lds_put(ex + Lds::kExchMat + flip<16>(wr_a), dz[1]);
    };
    // ... and dQ += dZ K.
    auto add_dq = [&](bool seen, lds_u8* kt, const u32x4 (&dz)[2]) {
      if (seen) {
        lds_u8* t0 = kt + tr_k;
        lds_u8* t1 = kt + flip<32>(tr_k) + 512;
        auto kc_op = [&](int i) { const int o = 1024 * (i / kDTiles) + (i % kDTiles) * Lds::kKvPanel; return tr_pair<T>(t0 + o, t1 + o); };
        vec8 b[4];
#pragma unroll
        for (int i = 0; i < 4; i++) b[i] = kc_op(i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2 * kDTiles; i++) {
          dqacc[i % kDTiles] = Elem<T>::mfma(as_vec8<T>(dz[i / kDTiles]), b[i & 3], dqacc[i % kDTiles]);
          if (i + 4 < 2 * kDTiles) b[i & 3] = kc_op(i + 4);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    // What the tile above left of block t is asked for, once it is there.
    auto request_above = [&](int t) {
      if (seen_count <= t) seen_count = wait_for(pred, t, lane);
      const float* src = part + (int64_t)t * (kPieces * 1024);
      asm volatile("s_nop 4\n\tglobal_load_dwordx4 %0, %4, %5 sc1\n\tglobal_load_dwordx4 %1, %4, %5 offset:1024 sc1\n\t"
                   "global_load_dwordx4 %2, %4, %5 offset:2048 sc1\n\tglobal_load_dwordx4 %3, %4, %5 offset:3072 sc1"
                   : "=&v"(c0), "=&v"(c1), "=&v"(c2), "=&v"(c3) : "v"(lane16), "s"(src) : "memory");
    };
    const int steps = kWide ? n : (n + 1) / 2;
    // The block of step t that this wave contracts.
    auto block_of = [&](int t) { return kWide ? t : 2 * t + (wave >> 2); };
    lds_barrier();
    for (int t = 0; t < steps; ++t) {
      asm volatile("; nothing in flight");
      const float prod_in = n_prod, prod_in2 = kWide ? 0.f : n_prod2;
      const int first = kWide ? t : 2 * t, last = kWide ? t : 2 * t + 1;      // the step's key blocks
      const bool seen = has_rows && kRowKeys * last <= last_seen;
      lds_u8* kt = lds + Lds::kKv + (last & (Lds::kBufs - 1)) * Lds::kKvBuf;
      lds_u8* ex = lds + Lds::kExch + (last & (Lds::kBufs - 1)) * Lds::kExchBuf;
      u32x4 dz[2];
      float r_prod, r_prod2;
      int r_count, count;
      if constexpr (kWide) {
        asm volatile("s_nop 4\n\tglobal_load_dword %0, %2, %4 sc1\n\tglobal_load_dword %1, %3, %5"
                     : "=&v"(r_count), "=&v"(r_prod) : "v"(0), "v"(row_c * 4), "s"(pred), "s"(product_at(t + 1)) : "memory");
      } else {
        asm volatile("s_nop 4\n\tglobal_load_dword %0, %2, %3\n\tglobal_load_dword %1, %2, %4"
                     : "=&v"(r_prod), "=&v"(r_prod2)
                     : "v"(row_c * 4), "s"(product_at(2 * t + 2)), "s"(product_at(2 * t + 3)) : "memory");
      }
      request_kv(t + 1);
      const int tn = late ? t - 1 : t, block = block_of(tn);      // contracted in this step
      const bool any = tn >= 0 && (kWide || block < n);
      // The key blocks that are complete are passed on: the stores of the last one left before this step's four loads and have arrived when the
      // first weights are there.  (Passed on at the end of the step, and the count of the tile above read at the start of it, that count was one too
      // small in 6 steps of 10 at head_dim 64, 1 to 2 of 10 at 128, and a wave spent 800 to 2300 cycles reading it again.  Training passes,
      // us before / after: 12 heads x 64, 16384 tokens in 10 sequences 415 / 405; 32 heads x 8 x 4096 x 128 4366 / 4298; 12 x 4 x 8192 x 128 3132 / 3106.)
      auto pass_on = [&] {
        vm_wait<4>();
        if (lane == 0) *flag = seen_count == kChainBroken ? kChainBroken : kWide ? block : block - 1;      // (the one before was this wave's last)
      };
      if constexpr (kWide) {
        front(kRowKeys * t, seen, kt, ex, prod_in, dz, pass_on);
        // (In flight: count, product, K and V in two parts, the flag.  3 would do and measured the same, 32 heads x 8 x 4096 4279 us either way;
        // 2 does not count on the flag.)
        asm volatile("s_waitcnt vmcnt(2)\n\tv_mov_b32 %0, %2\n\tv_readfirstlane_b32 %1, %3"
                     : "=&v"(n_prod), "=s"(count) : "v"(r_prod), "v"(r_count) : "memory");
      } else {
        const bool seen1 = has_rows && kRowKeys * first <= last_seen;
        front(kRowKeys * first, seen1, kt - Lds::kKvBuf, ex - Lds::kExchBuf, prod_in, dz, pass_on);
        add_dq(seen1, kt - Lds::kKvBuf, dz);
        front(kRowKeys * last, seen, kt, ex, prod_in2, dz, [&] {      // (at head_dim 128 K and V would be waited for as well: 0 to +2 %)
          asm volatile("s_nop 4\n\tglobal_load_dword %0, %1, %2 sc1" : "=&v"(r_count) : "v"(0), "s"(pred) : "memory");
        });
        asm volatile("s_waitcnt vmcnt(0)\n\tv_mov_b32 %0, %3\n\tv_mov_b32 %1, %4\n\tv_readfirstlane_b32 %2, %5"
                     : "=&v"(n_prod), "=&v"(n_prod2), "=s"(count) : "v"(r_prod), "v"(r_prod2), "v"(r_count) : "memory");
      }
      // What the tile above left of the block that is contracted next is asked for.
      seen_count = max(seen_count, count);
      if (has_pred && any) request_above(block);
      else c0 = c1 = c2 = c3 = f32x4{0.f, 0.f, 0.f, 0.f};
      add_dq(seen, kt, dz);
      // The rows of step t + 1 are in LDS before the barrier (behind them: the flag, and what the tile above left).
      if (!late || !any) {
        if (has_pred && any) vm_wait<5>(); else vm_wait<1>();
      }
      if (!late) lds_barrier();
      if (any) contract(block);
      if (late) lds_barrier();
    }
    if (late) {
      vm_wait<0>();
      const int block = block_of(steps - 1);
      if (kWide || block < n) {
        if (has_pred) request_above(block);
        contract(block);
      }
    }
    // The last results are passed on.
    vm_wait<0>();
    if (lane == 0) *flag = seen_count == kChainBroken ? kChainBroken : n;
    if (has_rows) {
      const RowSink<T> dq_sink = make_row_sink<T>((T*)p.dq.ptr + seq_id * p.dq.sb + head * p.dq.sh + tok0 * p.dq.st, p.dq.st, L, DH);
#pragma unroll
      for (int dt = 0; dt < kDTiles; dt++) store_acc_tile<T>(dq_sink, dqacc[dt], p.logit_scale, w_first, 32 * dt, half, col, DH);
    }
    read_lists();
    __syncthreads();
  }
}

// Clears a region of `n16` pieces of 16 bytes.
__global__ __launch_bounds__(256) void row_clear_kernel(u32x4* z, int64_t n16) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += (int64_t)gridDim.x * 256) z[i] = u32x4{0u, 0u, 0u, 0u};
}

template <typename T, int DH, bool kAddRem>
static hipError_t launch_row_t(const BwdParams& p, int max_tiles, hipStream_t stream) {
  static std::atomic<uint64_t> lds_done{0};
  int dev = 0, cus = 0;
  hipError_t e = device_cus(&dev, &cus);
  if (e != hipSuccess) return e;
  if ((e = raise_lds_limit(&bwd_row_kernel<T, DH, kAddRem>, lds_done, dev, RowLds<DH>::kBytes)) != hipSuccess) return e;
  const int64_t tiles = (int64_t)max_tiles * ((p.num_heads + 7) / 8);      // per queue, at most
  const int per_queue = (int)(tiles < cus / 8 ? tiles : cus / 8);
  hipLaunchKernelGGL((bwd_row_kernel<T, DH, kAddRem>), dim3((unsigned)(8 * per_queue)), dim3(kRowThreads), RowLds<DH>::kBytes, stream, p);
  return hipGetLastError();
}

// Whether the tensors and the device allow the backward on row tiles.
bool row_supported(const BwdParams& p) {
  int dev = 0, cus = 0;
  if (device_cus(&dev, &cus) != hipSuccess) return false;
  return p.load == kLoadAligned && (p.head_dim == 64 || p.head_dim == 128) && !p.wide_rows && cus >= 8;
}

hipError_t launch_row_clear(uint32_t* region, int64_t bytes, hipStream_t stream) {
  const int64_t n16 = bytes / 16, wgs = (n16 + 1023) / 1024;
  hipLaunchKernelGGL(row_clear_kernel, dim3((unsigned)(wgs < 256 ? wgs : 256)), dim3(256), 0, stream, (u32x4*)region, n16);
  return hipGetLastError();
}

template <int DH>
static hipError_t launch_row_dim(const BwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream) {
  if (p.add_rem) return dtype_is_f16 ? launch_row_t<_Float16, DH, true>(p, max_tiles, stream) : launch_row_t<__bf16, DH, true>(p, max_tiles, stream);
  return dtype_is_f16 ? launch_row_t<_Float16, DH, false>(p, max_tiles, stream) : launch_row_t<__bf16, DH, false>(p, max_tiles, stream);
}
hipError_t launch_bwd_row(const BwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream) {
  return p.head_dim == 128 ? launch_row_dim<128>(p, dtype_is_f16, max_tiles, stream) : launch_row_dim<64>(p, dtype_is_f16, max_tiles, stream);
}

}  // namespace sba
