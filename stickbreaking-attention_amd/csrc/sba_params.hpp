// Kernel parameter blocks shared by the host launcher and the device code.
#pragma once
#include <stdint.h>

namespace sba {

struct TensorRef {     // [batch,] head, token, head_dim; element strides; head_dim stride 1
  void* ptr;
  int64_t sb, sh, st;
};
struct VectorRef {     // [batch,] head, token
  void* ptr;
  int64_t sb, sh, st;
};

// Tile descriptor produced by the scheduler kernel.
struct Tile {
  int32_t seq_start;   // first token of the sequence in the packed token axis (0 in fixed-length mode)
  int32_t seq_len;
  int32_t origin;      // first query row (query tiles) or first key (key tiles), relative to the sequence
  int32_t seq_id;      // sequence index; selects the batch stride in fixed-length mode
  int64_t carry_base;  // first carry slot of the sequence within a head's plane (0 when no carries are laid out)
};
// What a row tile (backward on row tiles) has to know of a list in which its sequence's tiles need not follow each other.
struct Turn {
  int32_t first_slot;  // of its sequence, in a list that held each sequence's tiles together: number in place of a slot
  int32_t rank;        // sequences before this one in that list
};

// How the 16-bit kernels read rows of head_dim elements, by what the tensors allow:
//   kLoadAligned : head_dim is the kernel's width (64 or 128) and every row starts on a 16-byte boundary: 16-byte loads.
//   kLoadPadded  : any head_dim from 8 on, any alignment: 16-byte loads all the same (the memory pipe takes them at any
//                  element's address).  A chunk of 8 columns that head_dim cuts is loaded from column head_dim - 8 and shifted
//                  into place, so that no load leaves its row; chunks beyond head_dim ask for an address outside the buffer.
//                  The shift costs 12 vector-ALU instructions per 16 bytes where head_dim is no multiple of 8.
//   kLoadScalar  : what is left (head_dim below 8, or a sequence whose rows span 2 GiB): element by element.
enum : int { kLoadScalar = 0, kLoadAligned = 1, kLoadPadded = 2 };

// A count of handed-over blocks that says: all of them, but what was handed over is not to be had (a wait ran out further up).
constexpr int kChainBroken = 0x7fffffff;

// Slots of the scheduler's `counts` array.
enum : int { kCountQ = 0, kCountK = 1, kCountStatus = 2, kCountCovered = 3, kCountChained = 4, kCountApart = 5 };
// Values of counts[kCountStatus].
enum : int { kSchedOk = 0, kSchedBadCu = 1, kSchedCarryOverflow = 2, kSchedChainTimeout = 3 };

struct SchedParams {
  const void* cu;          // NULL: fixed-length mode
  int32_t cu_is_int64, cu_has_leading_zero;
  int32_t num_seqs;
  int32_t fixed_len;       // L in fixed-length mode
  int64_t total_tokens;    // T: rows of the packed token axis (L in fixed-length mode)
  int64_t carry_capacity;  // carry slots reserved per head
  int64_t row_capacity;    // key blocks reserved per head for what row tiles hand over (< 0: not to be checked)
  int32_t want_key_tiles;  // backward: also build the key-tile list
  int32_t carry_rows;      // > 0: also lay out the per-sequence carry offsets; a sequence with more rows than this voids the schedule
  Tile* q_tiles;           // query tiles (kBlockQ rows), heaviest first
  Tile* k_tiles;           // key tiles (key_tile keys), heaviest first
  int32_t* counts;         // [kCountQ] query tiles, [kCountK] key tiles, [kCountStatus], [kCountCovered] = tokens
                           // covered by sequences (rows at or beyond it belong to no sequence and are zero-filled); row tiles:
                           // [kCountChained] tiles at the head of the list, behind which every tile is its sequence's only one,
                           // [kCountApart] what says how many workgroups begin with those (apart_share)
  int64_t* carry_base;     // per sequence: first carry slot of the sequence (per head)
  int32_t* head_queue;     // backward: per-head cursor into the key-tile list, reset to 0 here
  int32_t num_heads;
  int32_t key_tile;        // keys per key tile (a multiple of 32; what the dK/dV kernel that will run sweeps)
  int32_t tiny;            // not kTinyNone: sequences of up to kTinyRows tokens get no key tiles
  Turn* k_turns;           // row tiles: beside k_tiles (else NULL)
  int32_t take_turns;      // row tiles: sequences whose tiles take turns in the list, up to kMostTurns (1, and in the scheduler kernel:
                           // each sequence's follow each other)
  uint32_t* zero_fill;     // optional: 16-byte aligned region cleared by the launch (the one-kernel backward's flags
  int64_t zero_bytes;      // and tags start every call at zero), a multiple of 16 bytes
  int32_t service;         // workgroups at the head of a forward launch that schedule and clear (0: a scheduler launch did)
};
// Most sequences of a packed batch whose tiles the forward's workgroups derive themselves (one lane each).  The derivation
// takes 5 instructions per sequence and wave behind a scan of the lanes, and replaces a launch of 8 us in front of the forward.
constexpr int kInlineSeqs = 64;

// Sequences of up to kTinyRows tokens have a backward of their own (sba_bwd_tiny.hip): none of a call, all, or those there are, beside the
// kernels of the longer ones, which then have no key tiles of them.
constexpr int kTinyRows = 64;
enum : int { kTinyNone = 0, kTinyAll = 1, kTinyApart = 2 };

constexpr int kRowTileRows = 256;      // query rows per tile of the backward on row tiles
// Key blocks of 32 that the row tiles of a sequence hand over, rounded up to whole tiles (none if it is a single tile).
__host__ __device__ inline int64_t row_blocks(int64_t len) { return len > kRowTileRows ? (len + kRowTileRows - 1) / kRowTileRows * (kRowTileRows / 32) : 0; }
// What a sequence's row tiles cost, in key blocks swept: those up to each tile's diagonal, and one per tile for its rows.  (A tile costs 2 to 5 blocks
// besides those, but one of a short sequence, with few waves at work, less per block: 64 tokens 2.9, 16384 tokens 265 per tile.)
__host__ __device__ inline uint64_t row_work(int64_t len) {
  const uint64_t tiles = (uint64_t)(len + kRowTileRows - 1) / kRowTileRows, blocks = (uint64_t)(len + 31) / 32;
  return tiles * (blocks + 1) - tiles * (tiles - (tiles > 0)) / 2 * (kRowTileRows / 32);
}
// Workgroups of a queue that begin with the sequences of one tile: those tiles' share of the work, to the nearest, where it is at least a fifth and
// the longest sequence alone is two thirds, all other chains a sixteenth (`share`, in 1024ths, else 0: one list, longest first).  The chain then has
// most workgroups all the time, and when the short tiles are used up the shortest of its own are left.  Where the chains are less, or
// several, long sweeps start when all else is done and run on alone; and a share of a few workgroups is too coarse.  Training passes at head_dim 128, us, one
// list / two by the share:
//    of 32 workgroups        8 heads                 16                32
//     8   one of 16384 beside 2048 of up to 64   2670 / 2613   5318 / 5183   10970 / 10481
//     9   one of 16384 beside 2048 of 64         2822 / 2797
//    10   one of 14182 beside 1564 of 72         2336 / 2320
//     9   one of 13000 beside 2000 of 30         1887 / 1858                  7394 /  7345
//     9   one of 12881 beside  819 of 119        1827 / 1846
//    12   one of 11000 beside 1500 of 64         1603 / 1577                  6177 /  6152
//    10   one of  9942 beside  419 of 163        1263 / 1244
// and where there is one list
//    32   one of  1024 beside 2048 of 64          949 / 1022   1895 / 2052
//    31   one of  2048 beside 2048 of 64          951 /  989   1875 /  1955
//    24   three of 1500 beside 300 of 100         301 /  329    589 /  645    1162 /  1271
//    10   four of 5000 beside 1000 of 40         1247 / 1268   2445 / 2490    4800 /  4905
//     4   one of 14267 beside  299 of 112        1768 / 1824
//     4   one of 11452 beside  143 of 254        1288 / 1316
//    19   one of  8192 beside 2048 of 64         1408 / 1402
__host__ __device__ inline int apart_share(uint64_t single, uint64_t chained, uint64_t longest) {
  const uint64_t all = single + chained;
  return single && 5 * single >= all && 3 * longest >= 2 * all && 16 * chained <= 16 * longest + all ? (int)((double)single / (double)all * 1024.) : 0;
}
__host__ __device__ inline int apart_workgroups(int wgs, int share) { return (wgs * share + 512) >> 10; }
// Its queue, of 8, for head 0 of the sequence with this rank (the list holds the longest first); head h's is (this + h) % 8.  If the heads do
// not fill the queues evenly, the fuller ones are others for the next sequence, in an order that goes forth and back (a Gray code).
__host__ __device__ inline int row_queue(int rank, int heads) { return heads & 7 ? ((rank ^ rank >> 1) * (heads & 7)) & 7 : 0; }

// Sequences of a batch whose row tiles take turns, at most.  The tiles of a group of sequences come by the number of keys they sweep, those with
// most first: tile t of n of the group's j-th sequence (the first has most tiles) is at place j + sum over the group of max(0, tiles - (n - t)),
// and the tile above it, t - 1, at a lower one.  (The rule and what it gives stand with take_turns in sba_api.hip.)
constexpr int kMostTurns = 8;

struct FwdParams {
  TensorRef q, k, v, o;
  VectorRef rem;
  float* row_stat;
  int64_t stat_sb, stat_sh;    // row_stat strides (token stride 1)
  float* carry;                // optional [head][slot]: running product per (row, key tile)
  const int64_t* carry_base;
  int64_t carry_head_stride;
  const Tile* tiles;           // NULL: the workgroups derive their tiles from `sched`
  const int32_t* counts;
  SchedParams sched;
  int32_t num_heads, head_dim;
  float scale_log2;            // logit_scale * log2(e)
  int32_t attend_current;
  int32_t load;                // kLoadAligned, kLoadPadded or kLoadScalar: how rows are read
  int32_t add_rem;             // write o + rem * v
  int32_t max_tiles;           // query-tile slots the launch provides per head (>= counts[kCountQ])
  int64_t total_tokens;        // packed mode: rows of the token axis; rows no sequence covers are zero-filled
  int32_t fp32_products;       // fp32 path: products on the fp32 matrix instruction throughout
};

// fp32 backward: operands split and laid out by a kernel in front (sba_f32.hip), [plane][head][piece of 32 rows].
struct LaidPlanes {
  char* base;                  // NULL: none
  int64_t pieces;              // per head and plane
  int64_t plane_pieces;        // per plane
  int64_t per_seq;             // fixed-length mode: pieces per sequence (else 0)
};
constexpr int kLaidPlanes = 4;

struct BwdParams {
  TensorRef q, k, v, d_o, dq, dk, dv;
  VectorRef d_rem;
  const Tile* q_tiles;
  const Tile* k_tiles;
  const Turn* k_turns;         // row tiles: beside k_tiles
  const int32_t* counts;
  const int64_t* carry_base;
  const float* carry;          // [head][slot]: the forward's running product per (row, 32-key sub-tile)
  float* prefix;               // [head][slot]: prefix sum of g over the keys below the sub-tile, per (row, sub-tile)
  int64_t carry_head_stride;   // carry slots reserved per head
  int32_t num_heads, head_dim;
  float scale_log2;
  float logit_scale;
  int32_t attend_current;
  int32_t load;                // as in FwdParams
  int32_t wide_rows;           // a row stride of 4 MiB or more
  int32_t split;               // dK/dV: too few key tiles to fill the chip
  int32_t tiny;                // kTinyNone, kTinyAll or kTinyApart
  // Fused remainder term (the forward wrote o + rem * v): d_rem_eff = d_rem + d_o . v per row, dv += rem * d_o.
  int32_t add_rem;
  const float* row_stat;       // log2(rem), fp32 [batch][head][token]
  int64_t stat_sb, stat_sh;
  int32_t wgs_per_head;        // persistent dK/dV workgroups per head
  int32_t* head_queue;         // per head: next key tile not yet taken (beyond the first wgs_per_head), zero at launch
  int64_t drem_sb;             // batch stride of drem_eff: the heads of THIS launch (row_stat's stride counts the caller's)
  float* drem_eff;             // workspace, (B, heads, T) fp32: the gradient of rem per row in fp32 (d_rem, plus
                               // d_o . v when add_rem), written by the dQ kernel and read by the dK/dV kernel
  int32_t max_tiles;           // query-tile slots the dQ launch provides per head
  int64_t total_tokens;        // packed mode: rows of the token axis; rows no sequence covers are zero-filled
  // What the key tiles (sba_bwd_chain.hip) or row tiles (sba_bwd_row.hip) of a (head, sequence) hand to each other.
  float* chain_dq;             // key tiles: [head][row][128] fp32, partial dQ of a row over the key tiles below the reader;
                               // row tiles: [head][key block of 32][32 x 256] fp32, partial dV and dK over the row tiles above
  uint32_t* chain_c;           // key tiles: [head][row] {fp32 C below the reader's tile, tag = index of the reader's tile};
                               // row tiles: [2][8], next tile not yet taken, per list and queue
  int32_t* chain_flags;        // [head][tile slot][8]: per wave, row (key) blocks whose partial result is complete
  int32_t* chain_head_xcc;     // [head] (row tiles: [queue]): XCC id + 1 of its first workgroup (0 = none yet); those on other XCDs leave
  int32_t* status;             // the scheduler's status word; the kernel raises it when a wait runs out
  int32_t wait_polls;          // polls after which a wait runs out: what depends on it comes out as NaN
  int64_t chain_rows;          // rows (row tiles: key blocks) per head in chain_dq / chain_c
  int32_t chain_by_slot;       // row tiles: a sequence's key blocks lie at 8 * its first slot of the list (else at 9/256 * its first token)
  int64_t chain_sb;            // fixed-length mode: rows per batch element (0 in packed mode)
  int32_t chain_tile_cap;      // key-tile slots per head in chain_flags
  int32_t fp32_products;       // as in FwdParams
  LaidPlanes laid;             // fp32
};

// One sequence's token range from cu_seqlens (cumulative sequence ends, optionally preceded by a 0).  Returns false
// when the entry is unusable: ends must be non-decreasing, within [0, total_tokens], and a leading entry must be 0.
// The reference reads the same two entries without any check (sb_varlen_fwd.py:283-288); here a bad entry voids the
// whole schedule instead of sending tiles outside the tensors.  Shared by the device scheduler and its host mirror.
__host__ __device__ inline bool seq_span(const void* cu, int is_int64, int leading_zero, int s, int64_t total_tokens,
                                         int32_t* start, int32_t* len) {
  const int idx = s + (leading_zero ? 1 : 0);
  const int64_t end = is_int64 ? ((const int64_t*)cu)[idx] : (int64_t)((const int32_t*)cu)[idx];
  const int64_t beg = idx == 0 ? 0 : (is_int64 ? ((const int64_t*)cu)[idx - 1] : (int64_t)((const int32_t*)cu)[idx - 1]);
  const bool ok = beg >= 0 && beg <= end && end <= total_tokens && !(leading_zero && s == 0 && beg != 0);
  *start = ok ? (int32_t)beg : 0;
  *len = ok ? (int32_t)(end - beg) : 0;
  return ok;
}

// Carry slots.  Carries are kept per (row, 32-key sub-tile): sub-tile U covers keys 32U .. 32U+31 of the
// sequence and is needed by the rows of query tiles U/4, U/4 + 1, ..., M-1 (M = query tiles of 128 rows the
// sequence rounds up to).  Slot of (sub-tile U, row i), i >= 128*(U/4):
//   carry_offset(U, M) + (i - 128*(U/4))
__host__ __device__ inline int64_t carry_offset(int64_t U, int64_t M) {
  const int64_t q = U >> 2, r = U & 3;
  const int64_t tri = 2 * q * (q - 1) + r * q;            // sum_{U' < U} floor(U'/4)
  return U * (M * 128) - 128 * tri;
}
// From a row's slot in sub-tile U to its slot in sub-tile U + 1 (or U + 4): a sweep steps from one to the next without the above, which is 20 scalar
// instructions.
__host__ __device__ inline int carry_step(int U, int M) { return 128 * (M - ((U + 1) >> 2)); }
__host__ __device__ inline int carry_step4(int U, int M) { return 128 * (4 * M - U - 1); }
__host__ __device__ inline int64_t carry_slots(int64_t M) { return 256 * M * (M + 1); }   // carry_offset(4M, M)

}  // namespace sba
