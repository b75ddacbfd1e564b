// Device-side scheduling: which tile a workgroup works on, from cu_seqlens.  Shared by the scheduler kernel and by the forward
// kernels, which derive their tile themselves where that is cheaper than a launch in front of them.
#pragma once
#include "sba_device.hpp"
#include "sba_params.hpp"

namespace sba {

// Returns false for an unusable cu_seqlens entry (see seq_span); the span is then empty.
__device__ __forceinline__ bool seq_bounds(const SchedParams& p, int s, int* start, int* len) {
  if (p.cu == nullptr) { *start = 0; *len = p.fixed_len; return true; }
  return seq_span(p.cu, p.cu_is_int64, p.cu_has_leading_zero, s, p.total_tokens, start, len);
}

// Sums over the lanes up to and including this one, and the greatest over a wave; exchanges between lanes are DPP moves (no LDS).
template <int kCtrl, int kRows>
__device__ __forceinline__ uint64_t dpp_or_0(uint64_t x) {
  const int lo = __builtin_amdgcn_update_dpp(0, (int)x, kCtrl, kRows, 0xf, false), hi = __builtin_amdgcn_update_dpp(0, (int)(x >> 32), kCtrl, kRows, 0xf, false);
  return (uint64_t)(uint32_t)lo | (uint64_t)(uint32_t)hi << 32;
}
template <int kCtrl, int kRows>
__device__ __forceinline__ int dpp_or_0(int x) { return __builtin_amdgcn_update_dpp(0, x, kCtrl, kRows, 0xf, false); }
template <typename V>
__device__ __forceinline__ V sum_up_to_lane(V x) {
  x += dpp_or_0<0x111, 0xf>(x);      // row_shr 1, 2, 4, 8: within 16 lanes
  x += dpp_or_0<0x112, 0xf>(x);
  x += dpp_or_0<0x114, 0xf>(x);
  x += dpp_or_0<0x118, 0xf>(x);
  x += dpp_or_0<0x142, 0xa>(x);      // row_bcast 15 into rows 1 and 3, 31 into rows 2 and 3
  x += dpp_or_0<0x143, 0xc>(x);
  return x;
}
template <typename V>
__device__ __forceinline__ V read_lane(V x, int lane) {
  if constexpr (sizeof(V) == 4) return __builtin_amdgcn_readlane(x, lane);
  else return (V)((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)x, lane) | (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(x >> 32), lane) << 32);
}
__device__ __forceinline__ uint64_t wave_sum(uint64_t x) { return read_lane(sum_up_to_lane(x), 63); }
__device__ __forceinline__ uint64_t wave_max(uint64_t x) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    const uint64_t y = __shfl_xor((unsigned long long)x, d);
    x = y > x ? y : x;
  }
  return x;
}

__device__ __forceinline__ int key_tiles(const SchedParams& p, int len) { return p.tiny && len <= kTinyRows ? 0 : (len + p.key_tile - 1) / p.key_tile; }

// Carry slots a sequence takes; one that is too long takes more than there are.  (Less than 2^24 sequences can be too long, so their sum does not
// overflow.  Forward, 8 heads x 128, 30 sequences: 15.6 us with and without this, 15.8 to 16.1 with a test and a field of its own.)
__device__ __forceinline__ uint64_t slots_of(const SchedParams& p, int len, int nq) { return len > p.carry_rows ? 1ull << 40 : carry_slots(nq); }

// A batch of at most kInlineSeqs sequences (or of equal ones) held by one wave, a sequence per lane.
struct SeqLanes {
  int start, len, nq;      // this lane's sequence, and its query tiles (0 beyond the last sequence)
  int status;              // kSchedOk, or why nothing is scheduled (uniform)
  int64_t carry_base;      // of this lane's sequence: the carry slots of those in front of it
};
__device__ __forceinline__ SeqLanes load_lanes(const SchedParams& p) {
  SeqLanes s{0, 0, 0, kSchedOk, 0};
  const int lane = threadIdx.x & 63;
  bool ok = true;
  if (lane < p.num_seqs) ok = seq_bounds(p, lane, &s.start, &s.len);
  s.nq = (s.len + kBlockQ - 1) / kBlockQ;
  if (__any(!ok)) s.status = kSchedBadCu;
  const uint64_t slots = slots_of(p, s.len, s.nq), upto = sum_up_to_lane(slots);
  s.carry_base = (int64_t)(upto - slots);
  if (s.status == kSchedOk && p.carry_rows && (int64_t)read_lane(upto, 63) > p.carry_capacity) s.status = kSchedCarryOverflow;
  if (s.status == kSchedOk && p.row_capacity >= 0 && (int64_t)wave_sum(row_blocks(s.len)) > p.row_capacity) s.status = kSchedCarryOverflow;
  return s;
}
// First slot of this lane's sequence in a list of `n` tiles per sequence: sequences with more query tiles first, then by
// index.  `total`: length of the list.
__device__ __forceinline__ int lane_slot(const SchedParams& p, const SeqLanes& s, int n, int* total = nullptr) {
  const int key = s.nq << 6 | (63 - (threadIdx.x & 63));      // (a sequence has less than 2^25 tiles)
  int before = 0;
  for (int j = 0; j < p.num_seqs; j++) {
    const int kj = __builtin_amdgcn_readlane(key, j), nj = __builtin_amdgcn_readlane(n, j);
    before += kj > key ? nj : 0;
  }
  if (total) *total = __builtin_amdgcn_readlane(sum_up_to_lane(n), 63);
  return before;
}

// The query tile in `slot`, derived by every wave for itself.  Returns false when the slot holds none: *covered then says from
// which token on rows belong to no sequence, *total how many slots do hold a tile.
__device__ __forceinline__ bool inline_q_tile(const SchedParams& p, int slot, Tile* t, int* total, int64_t* covered) {
  if (p.cu == nullptr) {
    const int nq = (p.fixed_len + kBlockQ - 1) / kBlockQ, seq = slot / nq;
    *total = nq * p.num_seqs;
    *covered = p.total_tokens;
    if (slot >= *total) return false;
    t->seq_start = 0; t->seq_len = p.fixed_len; t->seq_id = seq;
    t->origin = (nq - 1 - (slot - seq * nq)) * kBlockQ;
    t->carry_base = seq * carry_slots(nq);
    return true;
  }
  const SeqLanes s = load_lanes(p);
  *total = 0; *covered = 0;
  if (s.status != kSchedOk) return false;
  const int first = lane_slot(p, s, s.nq, total);
  *covered = __builtin_amdgcn_readlane(s.start + s.len, p.num_seqs - 1);
  const uint64_t mine = __ballot(slot >= first && slot < first + s.nq);
  if (!mine) return false;
  const int seq = __builtin_ctzll(mine);
  t->seq_start = __builtin_amdgcn_readlane(s.start, seq);
  t->seq_len = __builtin_amdgcn_readlane(s.len, seq);
  t->seq_id = seq;
  t->origin = (__builtin_amdgcn_readlane(s.nq, seq) - 1 - (slot - __builtin_amdgcn_readlane(first, seq))) * kBlockQ;
  t->carry_base = p.carry_rows ? read_lane(s.carry_base, seq) : 0;
  return true;
}

// The tile lists of a batch held by the lanes.  A wave of the workgroup lists every fourth sequence: a lane the tiles of its own one where they are
// few, the wave together those of a longer one.  (One sequence after the other, by the whole workgroup, took 0.6 us each, which was most of a
// training forward of up to 64 short sequences: forward kernel, 7 heads x 64, 64 sequences of 32 / 64 / 128 tokens 49 / 39 / 39 us, then, the sums of
// load_lanes by scans instead of loops as well, 23 / 10 / 13.)
constexpr int kLaneTiles = 4;      // query tiles of a sequence that a lane lists
__device__ __forceinline__ void list_lanes(const SchedParams& p, const SeqLanes& s, int first_q, int first_k, int nk, int* chained, int* apart) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6, turns = p.take_turns;
  if (wave == 0 && lane < p.num_seqs) p.carry_base[lane] = s.carry_base;

  // Row tiles: the group of sequences this lane's one takes turns with: its rank, where the group's first tiles begin, how many tiles they have.
  int rank = 0, start = 0, tiles[kMostTurns] = {};
  if (p.k_turns) {
    rank = lane_slot(p, s, nk > 0);
    const uint64_t here = __ballot(nk > 0);
    // (Empty sequences, which are in no group, come behind the others: every lane has a rank of its own.)
    const int place = nk > 0 ? rank : __builtin_popcountll(here) + __builtin_popcountll(~here & ((1ull << lane) - 1));
    const int nk_at = __builtin_amdgcn_ds_permute(place * 4, nk), first_at = __builtin_amdgcn_ds_permute(place * 4, first_k);      // by rank
    const int group = rank / turns * turns;
    start = __shfl(first_at, group & 63);
#pragma unroll
    for (int j = 0; j < kMostTurns; j++) {
      const int n = __shfl(nk_at, (group + j) & 63);
      tiles[j] = j < turns && group + j < 64 ? n : 0;
    }
    const int in_groups = (__builtin_popcountll(__ballot(nk > 1)) + turns - 1) / turns * turns;      // ranks of groups with a sequence of several tiles
    const uint64_t work = nk > 0 ? row_work(s.len) : 0;
    *chained = (int)wave_sum(nk > 0 && rank < in_groups ? nk : 0);
    *apart = apart_share(wave_sum(nk > 1 ? 0 : work), wave_sum(nk > 1 ? work : 0), wave_max(work));
  }

  auto list_keys = [&](Tile t, int i, int n, int k0, int mine, int from, const int (&of)[kMostTurns]) {
    t.origin = i * p.key_tile;
    int place = k0 + i;
    if (p.k_turns) {
      place = from + mine % turns;
#pragma unroll
      for (int j = 0; j < kMostTurns; j++) place += max(0, of[j] - (n - i));
      p.k_turns[place] = Turn{k0, mine};
    }
    p.k_tiles[place] = t;
  };
  const bool listed_here = lane % waves == wave && s.nq > 0;
  if (listed_here && s.nq <= kLaneTiles) {
    Tile t;
    t.seq_start = s.start; t.seq_len = s.len; t.seq_id = lane; t.carry_base = s.carry_base;
    for (int i = 0; i < s.nq; i++) { t.origin = (s.nq - 1 - i) * kBlockQ; p.q_tiles[first_q + i] = t; }
    for (int i = 0; i < nk; i++) list_keys(t, i, nk, first_k, rank, start, tiles);
  }
  for (uint64_t left = __ballot(listed_here && s.nq > kLaneTiles); left; left &= left - 1) {
    const int seq = __builtin_ctzll(left);
    const int nq = __builtin_amdgcn_readlane(s.nq, seq), n = __builtin_amdgcn_readlane(nk, seq), q0 = __builtin_amdgcn_readlane(first_q, seq),
              k0 = __builtin_amdgcn_readlane(first_k, seq), mine = __builtin_amdgcn_readlane(rank, seq), from = __builtin_amdgcn_readlane(start, seq);
    int of[kMostTurns];
#pragma unroll
    for (int j = 0; j < kMostTurns; j++) of[j] = __builtin_amdgcn_readlane(tiles[j], seq);
    Tile t;
    t.seq_start = __builtin_amdgcn_readlane(s.start, seq); t.seq_len = __builtin_amdgcn_readlane(s.len, seq); t.seq_id = seq;
    t.carry_base = read_lane(s.carry_base, seq);
    for (int i = lane; i < nq; i += 64) { t.origin = (nq - 1 - i) * kBlockQ; p.q_tiles[q0 + i] = t; }
    for (int i = lane; i < n; i += 64) list_keys(t, i, n, k0, mine, from, of);
  }
}

// The first `p.service` workgroups of a forward launch: number 0 leaves the status word and, when a backward will follow, that
// backward's tile lists; the others clear what it needs cleared.
__device__ __forceinline__ void forward_service(const SchedParams& p, int wg) {
  if (wg > 0) {
    const int64_t n16 = p.zero_bytes / 16, per = (n16 + p.service - 2) / (p.service - 1);
    const int64_t a = per * (wg - 1), b = a + per < n16 ? a + per : n16;
    u32x4* z = reinterpret_cast<u32x4*>(p.zero_fill);
    for (int64_t i = a + threadIdx.x; i < b; i += blockDim.x) z[i] = u32x4{0u, 0u, 0u, 0u};
    return;
  }
  SeqLanes s{0, p.fixed_len, (p.fixed_len + kBlockQ - 1) / kBlockQ, kSchedOk, 0};
  int total_q, total_k = 0, first_q = 0, first_k = 0, chained = 0, apart = 0;
  int64_t covered = p.total_tokens;
  if (p.cu == nullptr) {
    total_q = s.nq * p.num_seqs;
  } else {
    s = load_lanes(p);
    first_q = lane_slot(p, s, s.nq, &total_q);
    covered = __builtin_amdgcn_readlane(s.start + s.len, p.num_seqs - 1);
  }
  const bool ok = s.status == kSchedOk;
  if (p.want_key_tiles && ok) {
    const int nk = key_tiles(p, s.len);
    if (p.cu == nullptr) total_k = nk * p.num_seqs; else first_k = lane_slot(p, s, nk, &total_k);
    if (p.cu == nullptr) chained = nk > 1 ? total_k : 0;
    const int turns = p.take_turns;
    Tile t;
    t.seq_start = 0; t.seq_len = s.len;
    if (p.cu == nullptr) {
      for (int i = threadIdx.x; i < total_q; i += blockDim.x) {
        t.seq_id = i / s.nq; t.origin = (s.nq - 1 - i % s.nq) * kBlockQ; t.carry_base = t.seq_id * carry_slots(s.nq);
        p.q_tiles[i] = t;
      }
      for (int i = threadIdx.x; i < total_k; i += blockDim.x) {
        t.seq_id = i / nk; t.origin = i % nk * p.key_tile; t.carry_base = t.seq_id * carry_slots(s.nq);
        int place = i;
        if (p.k_turns) {      // (sequences of equal length)
          const int group = t.seq_id / turns * turns, members = min(turns, p.num_seqs - group);
          place = group * nk + i % nk * members + (t.seq_id - group);
          p.k_turns[place] = Turn{t.seq_id * nk, t.seq_id};
        }
        p.k_tiles[place] = t;
      }
      for (int i = threadIdx.x; i < p.num_seqs; i += blockDim.x) p.carry_base[i] = i * carry_slots(s.nq);
    } else {
      list_lanes(p, s, first_q, first_k, nk, &chained, &apart);
    }
  }
  if (p.want_key_tiles)
    for (int h = threadIdx.x; h < p.num_heads; h += blockDim.x) p.head_queue[h] = 0;
  if (threadIdx.x == 0) {
    p.counts[kCountQ] = ok ? total_q : 0;
    p.counts[kCountK] = total_k;
    p.counts[kCountStatus] = s.status;
    p.counts[kCountCovered] = ok ? (int32_t)covered : 0;
    p.counts[kCountChained] = chained;
    p.counts[kCountApart] = apart;
  }
}

// The query tile a forward workgroup works on: from the list the scheduler kernel left, or derived on the spot.  Returns false
// when there is none; *r0..*r1 are then the rows of no sequence this slot clears, if any.
__device__ __forceinline__ bool forward_tile(const FwdParams& p, int slot, int sub, int rows, Tile* t, int64_t* r0, int64_t* r1) {
  int total;
  int64_t covered;
  bool found;
  if (p.tiles) {
    total = p.counts[kCountQ];
    found = slot < total;
    if (found) *t = p.tiles[slot]; else covered = p.counts[kCountCovered];
  } else {
    found = inline_q_tile(p.sched, slot, t, &total, &covered);
  }
  if (found) {      // uniform, which the compiler does not see through the lane exchanges
    t->seq_start = __builtin_amdgcn_readfirstlane(t->seq_start); t->seq_len = __builtin_amdgcn_readfirstlane(t->seq_len);
    t->seq_id = __builtin_amdgcn_readfirstlane(t->seq_id); t->origin = __builtin_amdgcn_readfirstlane(t->origin);
    t->carry_base = (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)t->carry_base) |
                    (int64_t)__builtin_amdgcn_readfirstlane((int)(t->carry_base >> 32)) << 32;
    return true;
  }
  *r0 = covered + (int64_t)kBlockQ * (slot - total) + (int64_t)sub * rows;
  *r1 = *r0 + rows < p.total_tokens ? *r0 + rows : p.total_tokens;
  return false;
}

}  // namespace sba
