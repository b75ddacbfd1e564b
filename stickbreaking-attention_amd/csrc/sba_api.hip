// C ABI of libsba: argument validation, workspace layout and kernel launches.  See include/sba.h.
#include <hip/hip_runtime.h>

#include <atomic>

#include "../../include/sba.h"
#include "sba_internal.hpp"
#include "sba_params.hpp"

namespace sba {
hipError_t launch_sched(const SchedParams& p, int clear_wgs, hipStream_t stream);
hipError_t launch_fwd(const FwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream);
hipError_t launch_fwd_carry_only(const FwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream);
hipError_t launch_bwd_dq(const BwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream);
hipError_t launch_bwd_dkv(const BwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream);
int dkv_key_tile(const BwdParams& p);
bool chain_supported(const BwdParams& p);
hipError_t launch_bwd_chain(const BwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream);
bool row_supported(const BwdParams& p);
hipError_t launch_row_clear(uint32_t* region, int64_t bytes, hipStream_t stream);
hipError_t launch_bwd_row(const BwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream);
hipError_t launch_fwd_split(const FwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream);
hipError_t launch_fwd_split_carry_only(const FwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream);
hipError_t launch_bwd_dq_split(const BwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream);
hipError_t launch_bwd_dkv_split(const BwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream);
hipError_t launch_bwd_tiny(const BwdParams& p, int dtype_is_f16, int max_tiles, hipStream_t stream);
hipError_t launch_fwd_f32(const FwdParams& p, int64_t rows_heads, int64_t longest, int max_tiles, hipStream_t stream);
hipError_t launch_bwd_f32(const BwdParams& p, int64_t rows_heads, int64_t longest, int max_q_tiles, int max_k_tiles, hipStream_t stream);
bool fp32_products_only(int D, int64_t rows_heads, int64_t longest, float scale_log2);
}  // namespace sba

namespace {

constexpr double kLog2e = 1.4426950408889634;
constexpr int kBlockQ = 128, kBlockK = 64;

inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }
inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

struct Layout {
  int64_t max_q_tiles, max_k_tiles, carry_slots_per_head;
  // Offsets in the schedule, which a forward can prepare for the backward that follows it ...
  size_t off_counts, off_q_tiles, off_k_tiles, off_carry_base, off_queue, off_turns, sched_bytes;
  // ... and in the rest of a backward's workspace, which starts behind it.
  size_t off_prefix, off_drem, off_carry, rest_bytes;
  size_t fwd_bytes, bwd_bytes, carry_bytes;
  size_t laid_bytes;                        // fp32: behind the rest, where the workspace has them (see laid_pieces)
  size_t pass_bytes;                        // what ONE pass over these heads needs (bwd_bytes: what sba_bwd wants, see split_heads)
  // The backwards in which tiles hand partial sums to each other; these share the prefix plane's region (only one backward runs).
  enum Chain { kNone, kKeyTiles, kRowTiles };
  Chain chain;
  bool one_kernel;                          // what has to be cleared is cleared with the schedule (else by a kernel in front)
  int64_t chain_rows;                       // rows per head (key tiles), key blocks per head (row tiles)
  bool rows_by_slot;                        // see BwdParams::chain_by_slot; chain_rows is then checked on the device
  size_t off_chain_zero, chain_zero_bytes;  // {C, tag} per row or the queues, the flags and the XCC ids: cleared for every call
  size_t off_chain_c, off_chain_flags, off_chain_xcc;
  int64_t row_group;                        // row tiles: heads per launch (see plan), of which there are row_launches(heads)
  int64_t row_launches(int64_t heads) const { return cdiv(heads, row_group); }
  int32_t split_heads;                      // > 0: sba_bwd takes this many heads (a multiple of 8) through the one-kernel
                                            // backward and the rest through the two kernels
};

constexpr int64_t kRowTilesFrom = 64 << 10;      // rows x heads from which the backward on row tiles runs (see plan)

// Whether the 8 queues of the backward on row tiles, each fed to one XCD, hold about the same work, within 8/7 of the mean.  With a head
// count that is a multiple of 8 they do; else a queue may hold one head of a sequence more than another, which evens out over the
// sequences (row_queue) but for what the longest has more than the others: at most its share of all pairs, where the others are equal.
bool queues_even(int64_t heads, int64_t seqs, int64_t tokens, int64_t max_len) {
  if ((heads & 7) == 0) return true;
  int64_t units[8] = {0}, most = 0;
  const int64_t n = seqs < 8 ? seqs : 8;      // (the pattern repeats)
  for (int64_t r = 0; r < n; r++)
    for (int64_t h = 0; h < heads; h++) units[(sba::row_queue((int)r, (int)(heads & 7)) + h) & 7]++;
  for (int64_t u : units) most = u > most ? u : most;
  if (most * 7 > heads * n) return false;
  if (max_len * seqs <= 2 * tokens) return true;
  const double others = seqs > 1 ? (double)(tokens - max_len) / max_len : 0., longest = 1. / (1. + others * others / (double)(seqs > 1 ? seqs - 1 : 1));
  return ((double)(8 * cdiv(heads, 8)) / (double)heads - 1.) * longest <= 1. / 7;
}

// Rows per head, and the longest sequence as far as the caller says.
int64_t rows_of(const SbaArgs* a) { return a->cu_seqlens ? a->total_tokens : a->num_seqs * a->total_tokens; }
int64_t longest_of(const SbaArgs* a) { return a->max_seqlen > 0 && a->max_seqlen < a->total_tokens ? a->max_seqlen : a->total_tokens; }

// What the caller says no sequence has more rows than.
int64_t claimed_rows(const SbaArgs* a) {
  return a->cu_seqlens && a->max_seqlen > 0 && a->max_seqlen < a->total_tokens ? a->max_seqlen : a->total_tokens;
}
// What a schedule holds the caller to: a backward of tiny sequences alone leaves a longer one's gradients unwritten, and a forward that it follows
// is void as well.  By what both passes are told alike, and not by whether that backward will run (strides and backward_kernels have their say in it).
int32_t most_rows_of(const SbaArgs* a) {
  return a->dtype != SBA_F32 && a->head_dim >= 8 && claimed_rows(a) <= sba::kTinyRows ? sba::kTinyRows : 0x7fffffff;
}

// Which sequences the backward of those of up to kTinyRows tokens takes (`heads`: of the whole call, `load`: as rows can be read): all, where there are no others, and those
// there are, beside longer ones, where there may be many.  Backward, us, the other kernels / with it: 32 heads, 2048 of 1 to 64 tokens (and one of
// 64), head_dim 128 2138 / 919, 64 1060 / 468; 1000 of those, 80 1050 / 447; 8 heads, 1000 of up to 64 and one of 300, 64 134 / 63, 128 296 / 47;
// 32 heads, 2048 of up to 64 beside one of 16384 8070 / 7160; 8 heads, 300 uniform in 1 to 200 130 / 121, log-normal around 55 (80 .. 99 on average)
// 0.75 .. 1.0 of the time, none of them tiny (65 to 128) 0.94 .. 1.0.  Up to 64 sequences lose (1.0 .. 1.5) and so do 242 with 2 heads (1.03): one
// more launch, little to gain.
int tiny_of(const SbaArgs* a, int64_t heads, int load) {
  if (a->dtype == SBA_F32 || load == sba::kLoadScalar || a->backward_kernels == 2) return sba::kTinyNone;
  if (claimed_rows(a) <= sba::kTinyRows) return sba::kTinyAll;
  return a->cu_seqlens && a->num_seqs > sba::kInlineSeqs && a->num_seqs * heads >= 1024 && a->total_tokens / a->num_seqs < 128 ?
             sba::kTinyApart : sba::kTinyNone;
}

// A piece of 32 rows in all planes: three numbers of 2 bytes per element.
int64_t laid_piece_bytes(const SbaArgs* a) { return sba::kLaidPlanes * 32 * 6 * (int64_t)align_up(a->head_dim, 32); }
// Pieces of 32 rows per head of the planes of split operands that the fp32 backward works from (0: it splits as it goes).  Laying them out costs
// what 6 bytes per element and plane cost (12 heads x 128, 6143 tokens: 65 + 45 us), what it saves goes by the pairs, so the line is the mean length.
// Training passes, laid out / split as it goes, by the bytes of the planes, 1 to 32 heads, head_dims 16 to 128:
//   mean length     512           1024          2048          4096          8192
//   to 256 MB       0.94 .. 1.06  0.84 .. 1.00  0.79 .. 0.93  0.74 .. 0.92  0.72 .. 0.91
//   beyond          1.08 .. 1.16  0.98 .. 1.05  0.86 .. 0.96  0.83 .. 0.92  0.85 .. 0.94
// and 6143 tokens in sequences of 83 to 2048 (mean 680, 226 MB) 1.04.  None where the shape already says that the products are
// of fp32 numbers.  (Sizes go by shapes and flags alone: a logit scale beyond 709 and rows 64 MiB apart leave the planes unused.)
int64_t laid_pieces(const SbaArgs* a) {
  if (a->dtype != SBA_F32 || sba::fp32_products_only(a->head_dim, rows_of(a) * a->num_heads, longest_of(a), 1.f)) return 0;
  const int64_t T = a->total_tokens, B = a->num_seqs, mean = a->cu_seqlens ? T / B : T, pieces = a->cu_seqlens ? (T >> 5) + B + 1 : B * cdiv(T, 32);
  const int64_t bytes = pieces * a->num_heads * laid_piece_bytes(a);
  return mean >= (bytes <= (int64_t)256 << 20 ? 1024 : 2048) && bytes <= (int64_t)4 << 30 ? pieces : 0;
}

// `row_tiles`: a group of the heads of a call that runs the backward on row tiles, which the group then runs as well (and nothing else:
// there is no room for the two kernels' planes).
int plan(const SbaArgs* a, Layout* out, bool row_tiles = false) {
  if (a->num_heads <= 0 || a->num_seqs <= 0 || a->total_tokens <= 0) return SBA_ERR_SHAPE;
  if (a->head_dim < 1 || a->head_dim > 128) return SBA_ERR_HEAD_DIM;
  if (a->dtype != SBA_BF16 && a->dtype != SBA_F16 && a->dtype != SBA_F32) return SBA_ERR_DTYPE;
  if (a->total_tokens > (int64_t)1 << 30) return SBA_ERR_SHAPE;
  if ((a->recompute_carry != 0 && a->recompute_carry != 1) || a->carry_slots < 0 || a->row_blocks < 0) return SBA_ERR_SHAPE;
  if (a->backward_kernels < 0 || a->backward_kernels > 2) return SBA_ERR_SHAPE;
  if (a->recompute_carry && a->dtype == SBA_F32) return SBA_ERR_DTYPE;      // the fp32 path always keeps its products
  Layout L{};
  const int64_t T = a->total_tokens, B = a->num_seqs;
  const bool fixed = a->cu_seqlens == nullptr;
  int64_t max_len = (a->max_seqlen > 0 && a->max_seqlen < T) ? a->max_seqlen : T;
  if (fixed) {
    L.max_q_tiles = B * cdiv(T, kBlockQ);
    L.max_k_tiles = B * cdiv(T, kBlockK);
    L.carry_slots_per_head = B * sba::carry_slots(cdiv(T, kBlockQ));
  } else {
    L.max_q_tiles = cdiv(T, kBlockQ) + B;
    L.max_k_tiles = cdiv(T, kBlockK) + B;
    // sum_s 256 M_s (M_s + 1) with M_s <= L_s/128 + 1 and sum_s L_s^2 <= T * max_len
    L.carry_slots_per_head = cdiv(T * max_len, 64) + 6 * T + 512 * B;
  }
  // A caller that knows the lengths passes the exact count (sba_plan_host); the scheduler checks it on the device.
  // (Fixed-length mode knows its exact count above; a caller's figure is not needed there and is ignored.)
  if (a->carry_slots > 0 && !fixed) L.carry_slots_per_head = a->carry_slots;
  size_t off = 0;
  L.off_counts = off;      off = align_up(off + 256, 256);
  L.off_q_tiles = off;     off = align_up(off + (size_t)L.max_q_tiles * sizeof(sba::Tile), 256);
  L.off_carry_base = off;  off = align_up(off + (size_t)B * sizeof(int64_t), 256);
  L.fwd_bytes = off;
  L.off_k_tiles = off;     off = align_up(off + (size_t)L.max_k_tiles * sizeof(sba::Tile), 256);
  L.off_queue = off;       off = align_up(off + (size_t)a->num_heads * sizeof(int32_t), 256);      // per-head tile cursors
  L.carry_bytes = align_up((size_t)L.carry_slots_per_head * a->num_heads * sizeof(float), 256);
  size_t chain_bytes = 0;
  const int64_t rows = fixed ? B * T : T;
  // Left to choose (backward_kernels 0), a backward whose tiles hand partial sums to each other runs where it is the faster one.
  // Training passes at head_dim 128 on 256 compute units.  Row tiles (sba_bwd_row.hip) over the better of key tiles and the two
  // kernels, equal sequences of 32768 tokens in all:
  //   length     64           128          192, 256     384          512          768 .. 4096   8192, 16384
  //              0.98 .. 1.01 0.92 .. 0.96 0.80 .. 0.86 0.93 .. 0.96 0.82 .. 0.85 0.79 .. 0.85  0.77 .. 0.85    (8 to 32 heads)
  //   and over the two kernels alone: 96 tokens 0.91 .. 0.92, 64 1.00, 48 1.06 .. 1.08, 32 0.98 .. 1.01, 24 1.00 .. 1.02, 16 1.03,
  //   8 1.05, 8 to 64 1.01 .. 1.03: where no sequence has more than 64 the two kernels run.
  // A tile is 256 rows, so 64 K rows x heads give a tile to each compute unit.  Down there, by rows x heads:
  //   64 K       512 .. 1024 tokens 0.77 .. 0.96     2048 tokens 0.86 (4 sequences), 0.97 (2), 1.04 (1)
  //   32 K       512 tokens 0.82 .. 0.97             1024 tokens 0.97 (4 sequences), 1.22 (2 and 1)     2048 tokens 1.25
  // where a tile's sweep over its keys is the time of the call, and key tiles of 128 keys are the better ones of long sequences:
  // key tiles over the two kernels
  //   20 K .. 64 K, length x heads from 16 K on      0.79 .. 0.93        up to 256 tokens  0.91 .. 0.97
  //   < 20 K        1024 to 2048 tokens              1.10 .. 1.25        up to 256 tokens  0.92 .. 1.20, one launch for two
  //   12 K .. 64 K  up to 64 tokens                  1.07 .. 1.26
  // At head_dim 64 (against the two kernels; the tiles' element-wise work bounds it, and rows that a tile does not fill cost more):
  //   length     64           128          256          384          512          768, 1024    2048, 4096   8192, 16384
  //   64 K       1.00         1.00         0.90 .. 1.00 1.03         0.84 .. 0.89 0.80 .. 0.84 0.83 .. 0.92 0.88 .. 1.00
  //   128 .. 512 K 1.20 .. 1.47 1.05 .. 1.26 0.89 .. 1.01 1.02 .. 1.16 0.82 .. 0.99 0.78 .. 0.95 0.76 .. 0.89 0.68 .. 0.81
  //   32 K       0.99         0.92 .. 1.00 1.00         0.97         0.99         1.02 .. 1.19 1.15 .. 1.48
  // and ragged ones with a mean of 512 to 1061, 7 to 24 heads: one of 16384 beside 260 or 40 tokens 0.78 .. 0.85, 4 of 4096 beside 300
  // 0.86 .. 0.89, 3 of 5000 beside 64 0.81 .. 0.93, 8 of 2000 beside 20 0.86 .. 0.89, halves of 1000 and 24 0.78 .. 0.91, 12 of 1300 beside 8
  // 0.88 .. 0.96.
  const int64_t mean_len = fixed ? T : T / B, rows_heads = rows * a->num_heads, mean_heads = mean_len * a->num_heads;
  const bool chain_shape = a->dtype != SBA_F32 && a->head_dim == 128 && (a->num_heads & 7) == 0 && !a->add_remainder;
  if (row_tiles) {
    L.chain = Layout::kRowTiles;
  } else if (rows_heads >= kRowTilesFrom && a->dtype != SBA_F32 && ((a->head_dim == 128 && max_len > 64) || (a->head_dim == 64 && mean_len >= 512)) && a->backward_kernels != 1 && (chain_shape || a->backward_kernels == 0)) {
    // One kernel where its flags were cleared with the schedule ...
    L.one_kernel = chain_shape && (a->backward_kernels == 2 || (max_len <= 128 && mean_len > 96) ||
                                   (a->num_heads <= 32 && mean_heads >= 32 << 10 && max_len * a->num_heads <= 192 << 10));
    if (L.one_kernel || queues_even(a->num_heads, B, rows, max_len)) L.chain = Layout::kRowTiles;
  } else if (chain_shape && (a->backward_kernels == 2 ||
                             (a->backward_kernels == 0 && rows_heads < kRowTilesFrom &&
                              ((max_len <= 256 && (mean_len > 64 || rows_heads < 12 << 10)) ||
                               (a->num_heads <= 32 && rows_heads >= 20 << 10 && mean_heads >= 16 << 10))))) {
    L.chain = Layout::kKeyTiles;
    L.one_kernel = true;
  }
  if (L.chain == Layout::kKeyTiles) {
    L.chain_rows = rows;
    L.off_chain_zero = off;
    L.off_chain_c = off;      off = align_up(off + (size_t)a->num_heads * L.chain_rows * 8, 256);
    L.off_chain_flags = off;  off = align_up(off + (size_t)a->num_heads * L.max_k_tiles * 32, 256);
    L.off_chain_xcc = off;    off = align_up(off + (size_t)a->num_heads * 4, 256);
    L.chain_zero_bytes = off - L.off_chain_zero;
    chain_bytes = align_up((size_t)a->num_heads * L.chain_rows * 128 * sizeof(float), 256);
  }
  // Row tiles: the region that is cleared lies in the schedule, or (two kernels) in the rest.
  auto row_region = [&]() {
    L.off_chain_zero = off;
    L.off_chain_c = off;      off = align_up(off + L.row_launches(a->num_heads) * 64, 256);      // the queues, two lists each
    L.off_chain_xcc = off;    off = align_up(off + L.row_launches(a->num_heads) * 32, 256);
    L.off_chain_flags = off;  off = align_up(off + (size_t)a->num_heads * L.max_k_tiles * 32, 256);
    L.chain_zero_bytes = off - L.off_chain_zero;
  };
  if (L.chain == Layout::kRowTiles) {
    // Key blocks of 32 per head.  (Unknown lengths: every sequence that hands any over is longer than 256.)  One more than needed: heads
    // a power of two apart meet in the same cache sets (32 heads x 8 x 4096, one pass of the backward: 3405 us without it, 3385 with it).
    L.off_turns = off;       off = align_up(off + (size_t)(fixed ? B * cdiv(T, sba::kRowTileRows) : cdiv(T, sba::kRowTileRows) + B) * sizeof(sba::Turn), 256);
    L.rows_by_slot = fixed || a->row_blocks > 0;
    L.chain_rows = fixed ? B * sba::row_blocks(T) + 1 : a->row_blocks > 0 ? (int64_t)a->row_blocks + 1 : rows * 9 / 256 + 2;
    L.row_group = a->num_heads;
    const int64_t row_block = 2 * 32 * 4 * (int64_t)a->head_dim;      // bytes of a key block's dV and dK
    // Where most sequences hand nothing over, the heads go through in several launches, multiples of 8 (an equal share for each
    // queue) that still fill the chip twice: what is handed over takes its turns in the same memory (2048 short sequences and one of 16384,
    // 32 heads, 8 at a time: 11570 -> 10760 to 10990 us).
    if (mean_len < sba::kRowTileRows && max_len > sba::kRowTileRows) {
      const bool apart = tiny_of(a, a->num_heads, sba::kLoadAligned) == sba::kTinyApart;      // (the longest is then what surely is here)
      const int64_t group = align_up(cdiv(2 * kRowTilesFrom, apart ? max_len : rows), 8);
      if (group < a->num_heads) L.row_group = group;
    }
    chain_bytes = (size_t)L.row_group * L.chain_rows * row_block;
    if (L.one_kernel) row_region();
  }
  L.sched_bytes = off;
  off = 0;
  L.off_prefix = off;      off += L.carry_bytes > chain_bytes && !row_tiles ? L.carry_bytes : align_up(chain_bytes, 256);
  // d_rem + d_o . v per row (fp32), used when the remainder term is fused
  L.off_drem = off;        off = align_up(off + (size_t)a->num_heads * (size_t)T * (fixed ? (size_t)B : 1) * sizeof(float), 256);
  // the forward's products, rebuilt inside the backward when the caller did not keep them
  L.off_carry = off;       if (a->recompute_carry) off += L.carry_bytes;
  if (L.chain == Layout::kRowTiles && !L.one_kernel) row_region();
  L.rest_bytes = off;
  L.pass_bytes = L.sched_bytes + L.rest_bytes;
  L.laid_bytes = (size_t)(laid_pieces(a) * a->num_heads * laid_piece_bytes(a));
  L.bwd_bytes = L.pass_bytes + (a->backward_kernels == 1 ? 0 : L.laid_bytes);
  // A head count that is not a multiple of 8 (the reference's own benchmarks use 12) cannot run the one-kernel backward,
  // whose workgroups of a head must share an XCD.  Left to choose, sba_bwd then takes the largest multiple of 8 through
  // it and the remaining heads through the two kernels, one pass after the other on the stream -- where that pays: two
  // passes have two tails and two schedules, and on the reference's sweep (12 heads, 4 sequences) the split costs 12 %
  // at 4096 tokens and 2 % at 8192 and gains 4 % at 12288 and 16384.  The workspace must hold either pass.
  if (!row_tiles && a->backward_kernels == 0 && (a->num_heads & 7) != 0 && a->num_heads > 8 &&
      mean_len * (a->num_heads & ~7) >= (int64_t)12288 * 8) {
    SbaArgs c = *a;
    c.num_heads = a->num_heads & ~7;
    Layout L8;
    if (L.chain == Layout::kNone && plan(&c, &L8) == SBA_OK && L8.one_kernel) {
      L.split_heads = c.num_heads;
      if (L8.bwd_bytes > L.bwd_bytes) L.bwd_bytes = L8.bwd_bytes;
    }
  }
  *out = L;
  return SBA_OK;
}

size_t elem_size(int dtype) { return dtype == SBA_F32 ? 4 : 2; }

// How the kernels may read (and write) the rows of these tensors.  The fp32 ones address 32 rows at a time, which must span less
// than 2 GiB, or else go through pointers (kLoadScalar).  16-bit: buffer accesses need the rows of one sequence, and
// the rows of the last tiles beyond it, within 2 GiB (32-bit offsets from the sequence's first row); the aligned form also
// base pointers and row/head/batch strides that are 16-byte multiples, and a head_dim that fills the kernel.
template <size_t N>
int row_load(const SbaArgs* a, const SbaTensor* const (&tensors)[N]) {
  if (a->dtype == SBA_F32) {
    for (const SbaTensor* t : tensors)
      if (t->ptr && t->stride_token > (int64_t)1 << 24) return sba::kLoadScalar;
    return sba::kLoadPadded;
  }
  if (a->head_dim < 8) return sba::kLoadScalar;
  const bool fixed = a->cu_seqlens == nullptr;
  const int64_t max_rows = (a->max_seqlen > 0 && a->max_seqlen < a->total_tokens) ? a->max_seqlen : a->total_tokens;
  int load = a->head_dim == 64 || a->head_dim == 128 ? sba::kLoadAligned : sba::kLoadPadded;
  for (const SbaTensor* t : tensors) {
    if (!t->ptr) continue;
    const int64_t row_bytes = t->stride_token * 2;
    if (load == sba::kLoadAligned) {
      if (((uintptr_t)t->ptr & 15) || ((t->stride_token | t->stride_head | (fixed ? t->stride_batch : 0)) & 7)) load = sba::kLoadPadded;
      else if (max_rows * row_bytes >= ((int64_t)1 << 31)) return sba::kLoadScalar;
    }
    if (load == sba::kLoadPadded && (max_rows + 256) * row_bytes >= ((int64_t)1 << 31)) return sba::kLoadScalar;
  }
  return load;
}
// Whether a call is too small to fill the chip with tiles of 128 query rows (or key tiles): its kernels then split the keys (rows) of a
// workgroup's rows (keys) over the waves.  An unsplit workgroup's longest row costs what it does however many rows there are, about a third of
// which remains when it is split; split kernels stage K and V four times as often, and launch four times the workgroups, of which a
// short sequence's rows fill one.  So the line, in rows x heads, rises with the longest sequence up to a cap, a sequence counts as 32 rows more
// than it has, and rows count for less the shorter the mean is (tiles of long sequences run first, short ones beside them fill the gaps).
// The two kinds round a row's weights at different places, and the line has no step in it, so that a prompt keeps its rows' bits while it
// grows on one side of it, from the first token on.  Split / unsplit, us, training calls on 256 compute units:
//   rows x heads         16 K             32 K             64 K         128 K
//   head_dim 64   fwd    12.6 / 14.4      20.4 / 16.1      39 / 22     54 / 34    512 tokens
//                        23.0 / 40.3      36.8 / 41.1      57 / 51     92 / 84   2048
//                        56.6 / 145       84.6 / 146      137 / 178              8192
//                 dQ     13.2 / 18.5      22.3 / 19.4                             512
//                        31.0 / 57.7      51.0 / 59.2                            2048
//                        82.0 / 217      114  / 218      251 / 340 (head_dim 50) 8192
//                 dK/dV  14.3 / 24.0 (50)                 54 / 37 (50)            512
//                        38.4 / 82.9 (50) 62.6 / 104 (48 K)  111 / 115 (50)      2048
//   head_dim 128  fwd    18.4 / 19.0      30.0 / 21.1      67 / 29                512
//                        37.0 / 55.2      59.2 / 56.8     101 / 73               2048
//                        91.7 / 200      132  / 204                              8192
//                 dQ     25.1 / 23.4      43.1 / 25.4                             512
//                        43.7 / 73.3      98.6 / 76.2                            2048
//                        130  / 275      258  / 280                              8192
//   and of short sequences, head_dim 64, fwd / dQ: 64 of 32 tokens, 4 heads 16.2 / 8.3, 13.1 / 5.2; 200 of 64, 4 heads 22.4 / 10.2, 36.9 / 12.6;
//   64 of 192, 1 head 10.0 / 10.6; one of 3000 and 3 of 300, 7 heads 28.8 / 56.5, 38.5 / 85.1.
// The lines lose 0.2 % on average and 14 to 22 % at most against the better kernel of each of 500 batches (1 to 400 equal, uniform, log-normal
// sequences, or one long among short ones, of up to 8192 tokens; 1 to 200 K rows x heads; head_dims 50 to 128).  A line by rows x heads and the
// longest sequence alone, drawn when the kernels were slower, lost 9 to 17 %, mostly on short sequences.
// `heads` is the head count of the caller's call, also where the backward takes them through in groups: the groups then run the
// kernels, and give the bits, of one pass, and products are rebuilt by the kernel whose forward would have kept them.
bool below_line(const SbaArgs* a, int64_t heads, int64_t base, int64_t slope, int64_t cap) {
  const int64_t tokens = a->total_tokens * (a->cu_seqlens ? 1 : a->num_seqs), mean = tokens / a->num_seqs;
  const int64_t longest = a->max_seqlen > 0 && a->max_seqlen < a->total_tokens ? a->max_seqlen : a->total_tokens;
  const int64_t line = base + slope * longest;
  return heads * (tokens + 32 * (int64_t)a->num_seqs) * (mean + 2 * longest) < 3 * longest * (line < cap ? line : cap);
}
bool few_tiles_fwd(const SbaArgs* a, int64_t heads, int load) {
  if (a->dtype == SBA_F32 || load == sba::kLoadScalar) return false;
  return a->head_dim > 64 ? below_line(a, heads, 10 << 10, 19, 48 << 10) : below_line(a, heads, 13 << 10, 25, 65 << 10);
}
bool few_tiles_dq(const SbaArgs* a, int64_t heads, int load) {
  if (a->dtype == SBA_F32 || load == sba::kLoadScalar) return false;
  return a->head_dim > 64 ? below_line(a, heads, 9 << 10, 6, 48 << 10) : below_line(a, heads, 19 << 10, 18, 80 << 10);
}
// The same for dK/dV: below, head_dim up to 64 splits the rows over the waves, wider ones take key tiles of 64 instead of 128.  These are also the
// better ones of short sequences, however many: 64 keys / 128 keys, us, 256 K to 512 K rows x heads,
//   tokens          20            64            256           512           1024          4096
//   head_dim 80     269 / 576     160 / 330     222 / 270     174 / 199     484 / 501     797 / 750
//            105    341 / 632     252 / 395     330 / 334     232 / 228     638 / 587     983 / 821
//            128    271 / 291     389 / 411 (1 M)
bool few_key_tiles(const SbaArgs* a, int64_t heads, int load) {
  if (a->dtype == SBA_F32 || load == sba::kLoadScalar) return false;
  if (a->head_dim <= 64) return below_line(a, heads, 10 << 10, 60, 153 << 10);
  const int64_t tokens = a->total_tokens * (a->cu_seqlens ? 1 : a->num_seqs);
  return tokens * heads < 100 << 10 || tokens / a->num_seqs < (a->head_dim & 7 ? 400 : 1100);
}
// Row strides from 4 MiB on: the offsets of a row tile's rows beyond the sequence would not stay within 32 bits.
template <size_t N>
bool wide_rows(const SbaTensor* const (&tensors)[N]) {
  for (const SbaTensor* t : tensors)
    if (t->ptr && t->stride_token >= (int64_t)2 << 20) return true;
  return false;
}
int check_tensor(const SbaTensor& t, bool required, bool fixed) {
  if (!t.ptr) return required ? SBA_ERR_NULL : SBA_OK;
  if (t.stride_token < 0 || t.stride_head < 0 || (fixed && t.stride_batch < 0)) return SBA_ERR_STRIDE;
  return SBA_OK;
}
sba::TensorRef ref(const SbaTensor& t, bool fixed) { return sba::TensorRef{t.ptr, fixed ? t.stride_batch : 0, t.stride_head, t.stride_token}; }
sba::VectorRef vref(const SbaVector& t, bool fixed) { return sba::VectorRef{t.ptr, fixed ? t.stride_batch : 0, t.stride_head, t.stride_token}; }

// Sequences whose row tiles take turns, by the heads of a launch: four (head, sequence) per queue, as far as there are any.  One after the
// other, the last sequence's longest tile starts when all others are nearly done (12 heads x 4 x 8192: the fullest queue's last tile would
// end 15 % behind the mean by the keys swept, 7 % when they take turns).  The more take turns, the fewer tiles of a (head, sequence) run at the
// same time and find in the L2 what the tile above left.  Training passes, us, one after the other / two per queue / four / eight:
// 12 heads x 4 x 8192 x 128 3356 / 3368 / 3255 / 3260; 16 heads, 16384 tokens in 14 sequences 870 / 867 / 857 / 855; 12 heads x 64, 16384 tokens in 10
// 432 / 435 / 430 / 433; 32 heads x 8 x 4096 4465 / - / 4483 / 4560.  (Where a forward prepares the schedule, of up to 64 sequences or of equal ones.  The
// scheduler kernel, which lists the others and those of a backward that has to schedule for itself, keeps each sequence's tiles together.)
int take_turns(int64_t heads) {
  const int64_t n = 32 / heads;
  return (int)(n < 1 ? 1 : n > sba::kMostTurns ? sba::kMostTurns : n);
}

// What the scheduler is asked for: always the query tiles; `for_backward`: the key tiles as well, the tile cursors at zero and
// what the one-kernel backward needs cleared; `carry_rows` as in SchedParams.
sba::SchedParams sched_params(const SbaArgs* a, char* ws, const Layout& L, bool for_backward, int32_t carry_rows, int key_tile) {
  sba::SchedParams sp{};
  if (for_backward && L.one_kernel) {
    sp.zero_fill = (uint32_t*)(ws + L.off_chain_zero);
    sp.zero_bytes = (int64_t)L.chain_zero_bytes;
  }
  sp.cu = a->cu_seqlens;
  sp.cu_is_int64 = a->cu_is_int64;
  sp.cu_has_leading_zero = a->cu_has_leading_zero;
  sp.num_seqs = a->num_seqs;
  sp.fixed_len = (int32_t)a->total_tokens;
  sp.total_tokens = a->total_tokens;
  sp.carry_capacity = L.carry_slots_per_head;
  sp.row_capacity = for_backward && L.chain == Layout::kRowTiles && L.rows_by_slot && a->cu_seqlens && key_tile == sba::kRowTileRows ? a->row_blocks : -1;
  sp.want_key_tiles = for_backward ? 1 : 0;
  sp.carry_rows = carry_rows;
  sp.q_tiles = (sba::Tile*)(ws + L.off_q_tiles);
  sp.k_tiles = (sba::Tile*)(ws + L.off_k_tiles);
  sp.counts = (int32_t*)(ws + L.off_counts);
  sp.carry_base = (int64_t*)(ws + L.off_carry_base);
  sp.head_queue = (int32_t*)(ws + L.off_queue);
  sp.num_heads = a->num_heads;
  sp.key_tile = key_tile;
  sp.take_turns = 1;
  if (for_backward && L.chain == Layout::kRowTiles && key_tile == sba::kRowTileRows) {
    sp.k_turns = (sba::Turn*)(ws + L.off_turns);
    sp.take_turns = take_turns(L.row_group);
  }
  return sp;
}

// Workgroups that clear the region a schedule is asked to clear: one per 256 KiB, at most 64.
int clear_wgs(const sba::SchedParams& sp) {
  const int64_t n = (sp.zero_bytes + (256 << 10) - 1) / (256 << 10);
  return (int)(n > 64 ? 64 : n);
}

// Whether the dK/dV kernel of a call with few key tiles runs: the one-kernel backward, where it is laid out and the rows allow
// it, takes such calls itself.
bool split_keys(const SbaArgs* a, const Layout& L, int64_t heads, int load) {
  return !(L.chain != Layout::kNone && load == sba::kLoadAligned) && few_key_tiles(a, heads, load);
}

// Which of the chained backwards a pass runs: the one that is laid out, if the tensors and the device allow it.
Layout::Chain chain_of(const Layout& L, const sba::BwdParams& p) {
  if (L.chain == Layout::kKeyTiles && sba::chain_supported(p)) return L.chain;
  if (L.chain == Layout::kRowTiles && sba::row_supported(p)) return L.chain;
  return Layout::kNone;
}
// Keys per key tile (row tiles: rows per tile) of the schedule such a pass wants.
int key_tile_of(const Layout& L, const sba::BwdParams& p) {
  return chain_of(L, p) == Layout::kRowTiles ? sba::kRowTileRows : sba::dkv_key_tile(p);
}

// Keys per key tile of the backward that will follow a forward, as far as the forward's tensors tell.
int expected_key_tile(const SbaArgs* a, const Layout& L) {
  if (a->dtype == SBA_F32) return kBlockK;
  sba::BwdParams p{};
  p.head_dim = a->head_dim;
  p.load = row_load(a, {&a->q, &a->k, &a->v});
  p.wide_rows = wide_rows({&a->q, &a->k, &a->v});
  p.num_heads = a->num_heads;
  p.add_rem = a->add_remainder ? 1 : 0;
  p.split = split_keys(a, L, a->num_heads, p.load);
  return key_tile_of(L, p);
}
// ... and whether it will take tiny sequences by themselves.
int expected_tiny(const SbaArgs* a) { return tiny_of(a, a->num_heads, row_load(a, {&a->q, &a->k, &a->v})); }

}  // namespace

extern "C" {

int sba_version(void) { return SBA_VERSION; }

const char* sba_strerror(int status) {
  switch (status) {
    case SBA_OK: return "ok";
    case SBA_ERR_NULL: return "a required pointer is NULL";
    case SBA_ERR_DTYPE: return "unsupported dtype";
    case SBA_ERR_HEAD_DIM: return "head_dim must be in 1..128";
    case SBA_ERR_STRIDE: return "negative or unsupported stride";
    case SBA_ERR_ALIGN: return "tensor base pointer is not aligned to its element size";
    case SBA_ERR_SHAPE: return "sizes must be positive (and total_tokens <= 2^30)";
    case SBA_ERR_WORKSPACE: return "workspace missing, misaligned or too small";
    case SBA_ERR_LAUNCH: return "kernel launch failed";
    case SBA_ERR_TOO_LARGE: return "the problem needs more scratch than the library's static array holds";
    default: return "unknown status";
  }
}

int sba_workspace_bytes(const SbaArgs* args, size_t* fwd_bytes, size_t* bwd_bytes, size_t* carry_bytes) {
  if (!args) return SBA_ERR_NULL;
  Layout L;
  const int st = plan(args, &L);
  if (st != SBA_OK) return st;
  if (fwd_bytes) *fwd_bytes = L.fwd_bytes;
  if (bwd_bytes) *bwd_bytes = L.bwd_bytes;
  if (carry_bytes) *carry_bytes = L.carry_bytes;
  return SBA_OK;
}

int sba_plan_host(const SbaArgs* a, const void* cu_host, SbaPlan* out) {
  if (!a || !out) return SBA_ERR_NULL;
  if (a->num_seqs <= 0 || a->total_tokens <= 0 || a->total_tokens > (int64_t)1 << 30) return SBA_ERR_SHAPE;
  SbaPlan pl{};
  const int ac = a->attend_current ? 1 : 0;
  for (int s = 0; s < a->num_seqs; s++) {
    int32_t start = 0, len = (int32_t)a->total_tokens;
    if (cu_host && !sba::seq_span(cu_host, a->cu_is_int64, a->cu_has_leading_zero, s, a->total_tokens, &start, &len))
      pl.status = SBA_SCHED_BAD_CU_SEQLENS;
    const int64_t n = len, m = cdiv(n, kBlockQ);
    pl.query_tiles += m;
    pl.key_tiles += cdiv(n, kBlockK);
    pl.carry_slots += sba::carry_slots(m);
    pl.pairs += n * (n - 1) / 2 + (ac ? n : 0);
    if (len > pl.longest) pl.longest = len;
    pl.covered_tokens = cu_host ? (int64_t)start + len : a->total_tokens;
  }
  if (pl.status != SBA_SCHED_OK) {      // the device scheduler voids the whole schedule
    pl.query_tiles = pl.key_tiles = pl.carry_slots = pl.pairs = pl.covered_tokens = 0;
    pl.longest = 0;
  }
  *out = pl;
  return SBA_OK;
}

}  // extern "C"

namespace {

// Scratch of sba_fwd_static: the forward's tile schedule (counts, query-tile list, per-sequence carry offsets) kept in
// a device array of the library instead of a caller workspace.  Every GPU the library runs on holds its own copy
// until the process ends.  Host code never uses the array's name as an address: the device address is looked up
// once per device with hipGetSymbolAddress and that pointer is what the kernels receive.
constexpr size_t kStaticScratchBytes = SBA_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

int static_scratch(char** out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return SBA_ERR_LAUNCH;
  void* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!ptr) {
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return SBA_ERR_LAUNCH;
    g_scratch_ptr[dev].store(ptr, std::memory_order_release);
  }
  *out = (char*)ptr;
  return SBA_OK;
}

// The forward on a given workspace (the caller's, or the library's static scratch).  `for_backward`: the workspace holds
// sched_bytes and keeps the schedule of the backward that will follow.  `alone`: none will follow, whatever the arguments keep for one.
int fwd_on(const SbaArgs* a, char* ws, size_t ws_bytes, bool ws_is_static, bool for_backward, bool alone = false) {
  Layout L;
  int st = plan(a, &L);
  if (st != SBA_OK) return st;
  const bool fixed = a->cu_seqlens == nullptr;
  const size_t es = elem_size(a->dtype);
  if ((st = check_tensor(a->q, true, fixed)) || (st = check_tensor(a->k, true, fixed)) ||
      (st = check_tensor(a->v, true, fixed)) || (st = check_tensor(a->o, true, fixed)))
    return st;
  if (!a->rem.ptr || !a->row_stat) return SBA_ERR_NULL;
  for (const SbaTensor* t : {&a->q, &a->k, &a->v, &a->o})
    if (t->ptr && ((uintptr_t)t->ptr % es)) return SBA_ERR_ALIGN;
  if (ws_is_static && ws_bytes < L.fwd_bytes) return SBA_ERR_TOO_LARGE;
  if (!ws || ((uintptr_t)ws & 255) || ws_bytes < (for_backward ? L.sched_bytes : L.fwd_bytes)) return SBA_ERR_WORKSPACE;
  hipStream_t stream = (hipStream_t)a->stream;
  // The carry offsets are laid out (and the capacity and the lengths checked) when products are recorded, and also when the backward
  // will rebuild them: both passes then agree on whether the schedule stands.
  sba::FwdParams p{};
  p.sched = sched_params(a, ws, L, for_backward, !a->carry && !a->recompute_carry ? 0 : alone ? 0x7fffffff : most_rows_of(a),
                         for_backward ? expected_key_tile(a, L) : kBlockK);
  if (for_backward) p.sched.tiny = expected_tiny(a);
  if (fixed || a->num_seqs <= sba::kInlineSeqs) {
    p.sched.service = 1 + clear_wgs(p.sched);
  } else {
    if (sba::launch_sched(p.sched, clear_wgs(p.sched), stream) != hipSuccess) return SBA_ERR_LAUNCH;
    p.tiles = (const sba::Tile*)(ws + L.off_q_tiles);
  }
  p.q = ref(a->q, fixed); p.k = ref(a->k, fixed); p.v = ref(a->v, fixed); p.o = ref(a->o, fixed);
  p.rem = vref(a->rem, fixed);
  p.row_stat = a->row_stat;
  p.carry = a->carry;
  p.carry_base = (const int64_t*)(ws + L.off_carry_base);
  p.carry_head_stride = L.carry_slots_per_head;
  p.stat_sb = fixed ? (int64_t)a->num_heads * a->total_tokens : 0;
  p.stat_sh = a->total_tokens;
  p.counts = (const int32_t*)(ws + L.off_counts);
  p.num_heads = a->num_heads;
  p.head_dim = a->head_dim;
  p.scale_log2 = (float)((double)a->logit_scale * kLog2e);
  p.attend_current = a->attend_current ? 1 : 0;
  p.add_rem = a->add_remainder ? 1 : 0;
  p.max_tiles = (int32_t)L.max_q_tiles;
  p.total_tokens = a->total_tokens;
  p.load = row_load(a, {&a->q, &a->k, &a->v, &a->o});
  hipEvent_t* ev = (hipEvent_t*)a->trace_events;
  if (ev && hipEventRecord(ev[0], stream) != hipSuccess) return SBA_ERR_LAUNCH;
  hipError_t e = (a->dtype == SBA_F32) ? sba::launch_fwd_f32(p, rows_of(a) * a->num_heads, longest_of(a), (int)L.max_q_tiles, stream)
                 : few_tiles_fwd(a, a->num_heads, p.load) ? sba::launch_fwd_split(p, a->dtype == SBA_F16, (int)L.max_q_tiles, stream)
                                         : sba::launch_fwd(p, a->dtype == SBA_F16, (int)L.max_q_tiles, stream);
  if (e != hipSuccess) return SBA_ERR_LAUNCH;
  if (ev && hipEventRecord(ev[1], stream) != hipSuccess) return SBA_ERR_LAUNCH;
  return SBA_OK;
}

}  // namespace

extern "C" {

int sba_fwd(const SbaArgs* a) {
  if (!a) return SBA_ERR_NULL;
  return fwd_on(a, (char*)a->workspace, a->workspace_bytes, false, false);
}

int sba_fwd_static(const SbaArgs* a) {
  if (!a) return SBA_ERR_NULL;
  char* ws = nullptr;
  const int st = static_scratch(&ws);
  if (st != SBA_OK) return st;
  return fwd_on(a, ws, kStaticScratchBytes, true, false);
}

}  // extern "C"

namespace {

int bwd_load(const SbaArgs* a) { return row_load(a, {&a->q, &a->k, &a->v, &a->d_o, &a->dq, &a->dk, &a->dv}); }
bool bwd_wide_rows(const SbaArgs* a) { return wide_rows({&a->q, &a->k, &a->v, &a->d_o, &a->dq, &a->dk, &a->dv}); }
// Which backward one pass over the heads `a` describes runs, and whether that is one kernel.
Layout::Chain form_of(const SbaArgs* a, const Layout& L) {
  if (a->dtype == SBA_F32) return Layout::kNone;
  sba::BwdParams p{};
  p.load = bwd_load(a);
  p.wide_rows = bwd_wide_rows(a);
  p.head_dim = a->head_dim;
  p.num_heads = a->num_heads;
  p.add_rem = a->add_remainder ? 1 : 0;
  return chain_of(L, p);
}
bool bwd_is_one_kernel(const SbaArgs* a, const Layout& L) { return L.one_kernel && form_of(a, L) != Layout::kNone; }

// The heads of a call from h0 on, as a call of their own.
SbaArgs heads_from(const SbaArgs* a, int64_t h0, int64_t count) {
  SbaArgs c = *a;
  const int64_t es = (int64_t)elem_size(a->dtype);
  Layout L;
  c.num_heads = (int32_t)count;
  for (SbaTensor* t : {&c.q, &c.k, &c.v, &c.d_o, &c.dq, &c.dk, &c.dv})
    if (t->ptr) t->ptr = (char*)t->ptr + h0 * t->stride_head * es;
  if (c.d_rem.ptr) c.d_rem.ptr = (char*)c.d_rem.ptr + h0 * c.d_rem.stride_head * es;
  if (c.carry && plan(a, &L) == SBA_OK) c.carry += h0 * L.carry_slots_per_head;      // slots per head do not depend on the head count
  if (c.row_stat) c.row_stat += h0 * a->total_tokens;
  return c;
}

// How sba_bwd takes a call through: passes of `group` heads, one after the other on the stream, and a last one of those that are left.
struct Route {
  int64_t group;
  int32_t kernels, tail_kernels;            // SbaArgs.backward_kernels of a pass
  bool row_tiles, tail_row_tiles;           // a group of a call that runs the backward on row tiles, which the group then runs as well
};

// `group` heads on row tiles: enough tiles for the chip, spread over its XCDs (as for a call of its own, see plan).
bool row_group(const SbaArgs* a, int64_t group) {
  return rows_of(a) * group >= kRowTilesFrom && queues_even(group, a->num_seqs, rows_of(a), longest_of(a));
}

int route_of(const SbaArgs* a, Route* out) {
  Layout L;
  const int st = plan(a, &L);
  if (st != SBA_OK) return st;
  Route r{a->num_heads, a->backward_kernels, a->backward_kernels, false, false};
  if (L.split_heads > 0 && a->workspace_bytes >= L.bwd_bytes) {
    const SbaArgs c = heads_from(a, 0, L.split_heads);
    Layout L8;
    if (plan(&c, &L8) == SBA_OK && bwd_is_one_kernel(&c, L8)) {      // (the tensors and the device allow the one kernel)
      *out = Route{L.split_heads, a->backward_kernels, 1, false, false};
      return SBA_OK;
    }
  }
  if (a->workspace_bytes >= L.pass_bytes || a->num_heads == 1) {
    *out = r;
    return SBA_OK;
  }
  // A workspace smaller than the whole call needs: the heads are independent, so they go through in groups of as many
  // as fit (the per-head planes dominate the workspace).
  SbaArgs c = *a;
  auto fits = [&](int64_t heads, bool row_tiles) {
    Layout G;
    c.num_heads = (int32_t)heads;
    return plan(&c, &G, row_tiles) == SBA_OK && G.pass_bytes <= a->workspace_bytes;
  };
  // The largest head count whose layout fits: plan() grows with num_heads.
  auto largest = [&](bool row_tiles) {
    int64_t lo = 0, hi = a->num_heads;
    while (lo < hi) {
      const int64_t mid = (lo + hi + 1) / 2;
      if (fits(mid, row_tiles)) lo = mid; else hi = mid - 1;
    }
    return lo;
  };
  if (form_of(a, L) == Layout::kRowTiles) {
    // Groups of one sequence's few heads would leave XCDs without work (8 heads x 65536, one at a time: 32 of 256 compute units), groups of few
    // rows most of them: such groups run the two kernels, which use all of them.
    // Equal groups if they suit, else the largest with a remainder that suits too, else the largest, its remainder on the two kernels.
    const int64_t most = largest(true);
    auto rest_suits = [&](int64_t group) { return a->num_heads % group == 0 || row_group(a, a->num_heads % group); };
    auto rest_fits = [&](int64_t group) {
      c.backward_kernels = 1;
      const bool ok = rest_suits(group) || fits(a->num_heads % group, false);
      c.backward_kernels = a->backward_kernels;
      return ok;
    };
    int64_t group = most > 0 ? cdiv(a->num_heads, cdiv(a->num_heads, most)) : 0;
    if (group > 0 && !(row_group(a, group) && rest_suits(group))) {
      for (group = most; group > 0 && !(row_group(a, group) && rest_suits(group));) group--;
      if (group == 0)
        for (group = most; group > 0 && !(row_group(a, group) && rest_fits(group));) group--;
    }
    if (group > 0) {
      *out = Route{group, a->backward_kernels, rest_suits(group) ? a->backward_kernels : 1, true, rest_suits(group)};
      return SBA_OK;
    }
  }
  // (a call that would not run either of the chained backwards runs the two kernels in groups too)
  if (L.chain != Layout::kKeyTiles) r.kernels = c.backward_kernels = 1;
  const int64_t lo = largest(false);
  if (lo < 1) return SBA_ERR_WORKSPACE;
  r.group = cdiv(a->num_heads, cdiv(a->num_heads, lo));
  // The one-kernel backward's layout is the larger one and is only laid out for head counts it applies to, so a group
  // size below `lo` need not fit although `lo` does: every pass then takes the two-kernel backward, whose layout grows
  // with the head count and therefore fits.
  const int64_t tail = a->num_heads % r.group;
  if (!fits(r.group, false) || (tail > 0 && !fits(tail, false))) r.kernels = 1;
  r.tail_kernels = r.kernels;
  *out = r;
  return SBA_OK;
}

// The backward on row tiles, in the launches that the layout asks for: each has queues of its own, what is handed over takes turns.
hipError_t launch_row_tiles(const sba::BwdParams& whole, const Layout& L, bool f16, hipStream_t stream) {
  const int64_t launches = L.row_launches(whole.num_heads);
  for (int64_t i = 0; i < launches; i++) {
    sba::BwdParams p = whole;
    const int64_t h0 = i * L.row_group;
    p.num_heads = (int32_t)(whole.num_heads - h0 < L.row_group ? whole.num_heads - h0 : L.row_group);
    for (sba::TensorRef* t : {&p.q, &p.k, &p.v, &p.d_o, &p.dq, &p.dk, &p.dv}) t->ptr = (char*)t->ptr + h0 * t->sh * 2;
    if (p.d_rem.ptr) p.d_rem.ptr = (char*)p.d_rem.ptr + h0 * p.d_rem.sh * 2;
    if (p.row_stat) p.row_stat += h0 * p.stat_sh;
    p.carry += h0 * p.carry_head_stride;
    p.chain_c += 16 * i;
    p.chain_head_xcc += 8 * i;
    p.chain_flags += h0 * p.chain_tile_cap * 8;
    const hipError_t e = sba::launch_bwd_row(p, f16, (int)L.max_k_tiles, stream);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// One pass of the backward over the heads `a` describes (all of them, or one group of a larger call: `stat_heads` is
// the head count of the caller's row_stat array, `first`/`last` say which trace events this pass records).  `sched`: the
// schedule a forward left (the workspace is then the rest), or NULL to run the
// scheduler here.  `polls`: of a wait between tiles before it runs out (0: about half a second's).
int bwd_pass(const SbaArgs* a, int64_t stat_heads, bool first, bool last, char* sched = nullptr, bool row_tiles = false, int32_t polls = 0) {
  Layout L;
  int st = plan(a, &L, row_tiles);
  if (st != SBA_OK) return st;
  const bool fixed = a->cu_seqlens == nullptr;
  const size_t es = elem_size(a->dtype);
  if ((st = check_tensor(a->q, true, fixed)) || (st = check_tensor(a->k, true, fixed)) ||
      (st = check_tensor(a->v, true, fixed)) || (st = check_tensor(a->d_o, true, fixed)) ||
      (st = check_tensor(a->dq, true, fixed)) || (st = check_tensor(a->dk, true, fixed)) ||
      (st = check_tensor(a->dv, true, fixed)))
    return st;
  if (!a->carry && !a->recompute_carry) return SBA_ERR_NULL;
  if (a->add_remainder && !a->row_stat) return SBA_ERR_NULL;
  for (const SbaTensor* t : {&a->q, &a->k, &a->v, &a->d_o, &a->dq, &a->dk, &a->dv})
    if (t->ptr && ((uintptr_t)t->ptr % es)) return SBA_ERR_ALIGN;
  if (!a->workspace || ((uintptr_t)a->workspace & 255) || a->workspace_bytes < (sched ? L.rest_bytes : L.pass_bytes)) return SBA_ERR_WORKSPACE;
  hipStream_t stream = (hipStream_t)a->stream;

  char* const ws = sched ? sched : (char*)a->workspace;
  char* const rest = sched ? (char*)a->workspace : ws + L.sched_bytes;
  sba::BwdParams p{};
  p.q = ref(a->q, fixed); p.k = ref(a->k, fixed); p.v = ref(a->v, fixed);
  p.d_o = ref(a->d_o, fixed);
  p.dq = ref(a->dq, fixed); p.dk = ref(a->dk, fixed); p.dv = ref(a->dv, fixed);
  p.d_rem = vref(a->d_rem, fixed);
  p.q_tiles = (const sba::Tile*)(ws + L.off_q_tiles);
  p.k_tiles = (const sba::Tile*)(ws + L.off_k_tiles);
  if (L.chain == Layout::kRowTiles) p.k_turns = (const sba::Turn*)(ws + L.off_turns);
  p.counts = (const int32_t*)(ws + L.off_counts);
  p.carry_base = (const int64_t*)(ws + L.off_carry_base);
  p.carry = a->recompute_carry ? (const float*)(rest + L.off_carry) : a->carry;
  p.prefix = (float*)(rest + L.off_prefix);
  p.carry_head_stride = L.carry_slots_per_head;
  p.num_heads = a->num_heads;
  p.head_dim = a->head_dim;
  p.scale_log2 = (float)((double)a->logit_scale * kLog2e);
  p.logit_scale = a->logit_scale;
  p.attend_current = a->attend_current ? 1 : 0;
  p.add_rem = a->add_remainder ? 1 : 0;
  p.row_stat = a->row_stat;
  p.stat_sb = fixed ? stat_heads * a->total_tokens : 0;
  p.stat_sh = a->total_tokens;
  p.drem_sb = fixed ? (int64_t)a->num_heads * a->total_tokens : 0;
  p.drem_eff = (float*)(rest + L.off_drem);
  p.head_queue = (int32_t*)(ws + L.off_queue);
  p.max_tiles = (int32_t)L.max_q_tiles;
  p.total_tokens = a->total_tokens;
  p.load = bwd_load(a);
  p.wide_rows = bwd_wide_rows(a);
  p.split = split_keys(a, L, stat_heads, p.load);
  p.tiny = tiny_of(a, stat_heads, p.load);
  // One kernel (the key tiles of a sequence hand C and partial dQ to each other) where it applies, else dQ then dK/dV.
  const Layout::Chain chain = a->dtype == SBA_F32 ? Layout::kNone : chain_of(L, p);
  if (row_tiles && chain != Layout::kRowTiles) return SBA_ERR_WORKSPACE;      // (route_of asked)
  char* const cleared = L.one_kernel ? ws : rest;
  if (chain != Layout::kNone) {
    p.chain_c = (uint32_t*)(cleared + L.off_chain_c);
    p.chain_flags = (int32_t*)(cleared + L.off_chain_flags);
    p.chain_head_xcc = (int32_t*)(cleared + L.off_chain_xcc);
    p.chain_dq = (float*)(rest + L.off_prefix);
    p.status = (int32_t*)(ws + L.off_counts) + sba::kCountStatus;
    p.wait_polls = polls > 0 ? polls : chain == Layout::kRowTiles ? 1 << 20 : 1 << 17;
    p.chain_rows = L.chain_rows;
    p.chain_by_slot = L.rows_by_slot ? 1 : 0;
    p.chain_sb = fixed ? a->total_tokens : 0;
    p.chain_tile_cap = (int32_t)L.max_k_tiles;
  }
  // The key-tile list is built for the dK/dV kernel that will run.
  const int key_tile = a->dtype == SBA_F32 ? kBlockK : key_tile_of(L, p);
  if (!sched) {
    sba::SchedParams sp = sched_params(a, ws, L, true, most_rows_of(a), key_tile);
    sp.tiny = p.tiny;
    if (sba::launch_sched(sp, clear_wgs(sp), stream) != hipSuccess) return SBA_ERR_LAUNCH;
  }
  hipEvent_t* ev = (hipEvent_t*)a->trace_events;
  if (ev && first && hipEventRecord(ev[0], stream) != hipSuccess) return SBA_ERR_LAUNCH;
  if (a->dtype == SBA_F32) {
    if (L.laid_bytes > 0 && p.load != sba::kLoadScalar && a->workspace_bytes >= (sched ? 0 : L.sched_bytes) + L.rest_bytes + L.laid_bytes) {
      const int64_t pieces = laid_pieces(a);
      p.laid = sba::LaidPlanes{rest + L.rest_bytes, pieces, pieces * a->num_heads, fixed ? cdiv(a->total_tokens, 32) : 0};
    }
    if (sba::launch_bwd_f32(p, rows_of(a) * stat_heads, longest_of(a), (int)L.max_q_tiles, (int)L.max_k_tiles, stream) != hipSuccess) return SBA_ERR_LAUNCH;
    if (ev && last && (hipEventRecord(ev[1], stream) != hipSuccess || hipEventRecord(ev[2], stream) != hipSuccess)) return SBA_ERR_LAUNCH;
    return SBA_OK;
  }
  if (a->recompute_carry) {
    // O(L) state between the passes: the products the forward would have recorded are rebuilt from q and k by the
    // forward kernel stripped of everything else (timed with the dQ kernel by trace_events).
    sba::FwdParams f{};
    f.q = p.q; f.k = p.k; f.v = p.v; f.o = p.q;
    f.carry = (float*)(rest + L.off_carry);
    f.carry_base = p.carry_base;
    f.carry_head_stride = L.carry_slots_per_head;
    f.tiles = p.q_tiles;
    f.counts = p.counts;
    f.num_heads = a->num_heads;
    f.head_dim = a->head_dim;
    f.scale_log2 = p.scale_log2;
    f.attend_current = p.attend_current;
    f.max_tiles = (int32_t)L.max_q_tiles;
    f.total_tokens = a->total_tokens;
    f.load = row_load(a, {&a->q, &a->k});
    if ((few_tiles_fwd(a, stat_heads, f.load) ? sba::launch_fwd_split_carry_only(f, a->dtype == SBA_F16, (int)L.max_q_tiles, stream)
                                          : sba::launch_fwd_carry_only(f, a->dtype == SBA_F16, (int)L.max_q_tiles, stream)) != hipSuccess)
      return SBA_ERR_LAUNCH;
  }
  if (p.tiny != sba::kTinyNone) {
    if (sba::launch_bwd_tiny(p, a->dtype == SBA_F16, (int)L.max_q_tiles, stream) != hipSuccess) return SBA_ERR_LAUNCH;
    if (p.tiny == sba::kTinyAll) {
      if (ev && last && (hipEventRecord(ev[1], stream) != hipSuccess || hipEventRecord(ev[2], stream) != hipSuccess)) return SBA_ERR_LAUNCH;
      return SBA_OK;
    }
  }
  if (chain != Layout::kNone) {
    if (!L.one_kernel && sba::launch_row_clear((uint32_t*)(cleared + L.off_chain_zero), (int64_t)L.chain_zero_bytes, stream) != hipSuccess)
      return SBA_ERR_LAUNCH;
    if (ev && last && hipEventRecord(ev[1], stream) != hipSuccess) return SBA_ERR_LAUNCH;
    if (chain == Layout::kRowTiles) {
      if (launch_row_tiles(p, L, a->dtype == SBA_F16, stream) != hipSuccess) return SBA_ERR_LAUNCH;
    } else if (sba::launch_bwd_chain(p, a->dtype == SBA_F16, (int)L.max_k_tiles, stream) != hipSuccess) {
      return SBA_ERR_LAUNCH;
    }
    if (ev && last && hipEventRecord(ev[2], stream) != hipSuccess) return SBA_ERR_LAUNCH;
    return SBA_OK;
  }
  const bool f16 = a->dtype == SBA_F16;
  if ((few_tiles_dq(a, stat_heads, p.load) ? sba::launch_bwd_dq_split(p, f16, (int)L.max_q_tiles, stream) : sba::launch_bwd_dq(p, f16, (int)L.max_q_tiles, stream)) != hipSuccess)
    return SBA_ERR_LAUNCH;
  if (ev && last && hipEventRecord(ev[1], stream) != hipSuccess) return SBA_ERR_LAUNCH;
  if ((p.split && a->head_dim <= 64 ? sba::launch_bwd_dkv_split(p, f16, (int)L.max_k_tiles, stream)
                                    : sba::launch_bwd_dkv(p, f16, (int)L.max_k_tiles, stream)) != hipSuccess)
    return SBA_ERR_LAUNCH;
  if (ev && last && hipEventRecord(ev[2], stream) != hipSuccess) return SBA_ERR_LAUNCH;
  return SBA_OK;
}


}  // namespace

extern "C" {

int sba_bwd_kernels(const SbaArgs* a) {
  if (!a) return SBA_ERR_NULL;
  Layout L;
  const int st = plan(a, &L);
  if (st != SBA_OK) return st;
  const int tiny = tiny_of(a, a->num_heads, bwd_load(a));
  return tiny == sba::kTinyAll ? 1 : (bwd_is_one_kernel(a, L) ? 1 : 2) + (tiny == sba::kTinyApart ? 1 : 0);
}

int sba_bwd(const SbaArgs* a) {
  if (!a) return SBA_ERR_NULL;
  Route r;
  int st = route_of(a, &r);
  if (st != SBA_OK) return st;
  for (int64_t h0 = 0; h0 < a->num_heads; h0 += r.group) {
    const bool tail = a->num_heads - h0 < r.group;
    SbaArgs c = heads_from(a, h0, tail ? a->num_heads - h0 : r.group);
    c.backward_kernels = tail ? r.tail_kernels : r.kernels;
    if ((st = bwd_pass(&c, a->num_heads, h0 == 0, h0 + r.group >= a->num_heads, nullptr, tail ? r.tail_row_tiles : r.row_tiles)) != SBA_OK) return st;
  }
  return SBA_OK;
}

}  // extern "C"

namespace sba {

int prepared_bytes(const SbaArgs* a, Prepared* out) {
  Layout L;
  const int st = plan(a, &L);
  if (st != SBA_OK) return st;
  *out = Prepared{L.sched_bytes, L.rest_bytes, L.laid_bytes, L.carry_bytes, L.one_kernel};
  return SBA_OK;
}

int forward_prepared(const SbaArgs* a) { return fwd_on(a, (char*)a->workspace, a->workspace_bytes, false, true); }
int forward_alone(const SbaArgs* a) { return fwd_on(a, (char*)a->workspace, a->workspace_bytes, false, false, true); }

bool prepared_fits(const SbaArgs* a) {
  Layout L;
  if (plan(a, &L) != SBA_OK || L.split_heads > 0) return false;
  BwdParams p{};
  p.head_dim = a->head_dim;
  p.load = bwd_load(a);
  p.wide_rows = bwd_wide_rows(a);
  p.num_heads = a->num_heads;
  p.add_rem = a->add_remainder ? 1 : 0;
  p.split = split_keys(a, L, a->num_heads, p.load);
  return a->dtype == SBA_F32 || (key_tile_of(L, p) == expected_key_tile(a, L) && tiny_of(a, a->num_heads, p.load) == expected_tiny(a));
}

int backward_route(const SbaArgs* a, BackwardRoute* out) {
  Route r;
  Layout L;
  const int st = route_of(a, &r);
  if (st != SBA_OK) return st;
  SbaArgs c = heads_from(a, 0, r.group);
  c.backward_kernels = r.kernels;
  if (plan(&c, &L, r.row_tiles) != SBA_OK) return SBA_ERR_SHAPE;
  const Layout::Chain chain = form_of(&c, L);
  *out = BackwardRoute{tiny_of(a, a->num_heads, bwd_load(a)) == sba::kTinyAll ? kBwdTiny : chain == Layout::kRowTiles ? kBwdRowTiles : chain == Layout::kKeyTiles ? kBwdKeyTiles : kBwdTwoKernels, (int32_t)r.group};
  return SBA_OK;
}

int backward_with_polls(const SbaArgs* a, int32_t polls) { return bwd_pass(a, a->num_heads, true, true, nullptr, false, polls); }

int backward_prepared(const SbaArgs* a, void* sched) { return bwd_pass(a, a->num_heads, true, true, (char*)sched); }

}  // namespace sba
