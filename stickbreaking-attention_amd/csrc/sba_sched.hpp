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

// A batch of at most kInlineSeqs sequences (or of equal ones) held by one wave, a sequence per lane.
struct SeqLanes {
  int start, len, nq;      // this lane's sequence, and its query tiles (0 beyond the last sequence)
  int status;              // kSchedOk, or why nothing is scheduled (uniform)
};
__device__ __forceinline__ SeqLanes load_lanes(const SchedParams& p) {
  SeqLanes s{0, 0, 0, kSchedOk};
  const int lane = threadIdx.x & 63;
  bool ok = true;
  if (lane < p.num_seqs) ok = seq_bounds(p, lane, &s.start, &s.len);
  s.nq = (s.len + kBlockQ - 1) / kBlockQ;
  if (__any(!ok)) s.status = kSchedBadCu;
  if (s.status == kSchedOk && p.want_carry_base) {
    int64_t slots = 0;
    for (int j = 0; j < p.num_seqs; j++) slots += carry_slots(__builtin_amdgcn_readlane(s.nq, j));
    if (slots > p.carry_capacity) s.status = kSchedCarryOverflow;
  }
  if (s.status == kSchedOk && p.row_capacity >= 0) {
    int64_t blocks = 0;
    for (int j = 0; j < p.num_seqs; j++) blocks += row_blocks(__builtin_amdgcn_readlane(s.len, j));
    if (blocks > p.row_capacity) s.status = kSchedCarryOverflow;
  }
  return s;
}
// First slot of this lane's sequence in a list of `n` tiles per sequence: sequences with more query tiles first, then by
// index.  `total`: length of the list.
__device__ __forceinline__ int lane_slot(const SchedParams& p, const SeqLanes& s, int n, int* total = nullptr) {
  const int lane = threadIdx.x & 63;
  int before = 0, sum = 0;
  for (int j = 0; j < p.num_seqs; j++) {
    const int qj = __builtin_amdgcn_readlane(s.nq, j), nj = __builtin_amdgcn_readlane(n, j);
    before += qj > s.nq || (qj == s.nq && j < lane) ? nj : 0;
    sum += nj;
  }
  if (total) *total = sum;
  return before;
}
__device__ __forceinline__ int64_t lane_carry_base(const SeqLanes& s, int seq) {
  int64_t base = 0;
  for (int j = 0; j < seq; j++) base += carry_slots(__builtin_amdgcn_readlane(s.nq, j));
  return base;
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
  t->carry_base = p.want_carry_base ? lane_carry_base(s, seq) : 0;
  return true;
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
  SeqLanes s{0, p.fixed_len, (p.fixed_len + kBlockQ - 1) / kBlockQ, kSchedOk};
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
    const int nk = (s.len + p.key_tile - 1) / p.key_tile;
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
      t.carry_base = 0;
      int rank = 0;      // of this lane's sequence
      if (p.k_turns) {
        rank = lane_slot(p, s, nk > 0);
        const int groups = (__builtin_popcountll(__ballot(nk > 1)) + turns - 1) / turns;      // with a sequence of several tiles
        uint64_t work[2] = {0, 0}, longest = 0;
        for (int seq = 0; seq < p.num_seqs; seq++) {
          const int n = __builtin_amdgcn_readlane(nk, seq);
          if (__builtin_amdgcn_readlane(rank, seq) < groups * turns) chained += n;
          const uint64_t of_seq = row_work(__builtin_amdgcn_readlane(s.len, seq));
          work[n > 1] += of_seq;
          longest = of_seq > longest ? of_seq : longest;
        }
        apart = apart_share(work[0], work[1], longest);
      }
      for (int seq = 0; seq < p.num_seqs; seq++) {
        const int nq = __builtin_amdgcn_readlane(s.nq, seq), n = __builtin_amdgcn_readlane(nk, seq);
        const int q0 = __builtin_amdgcn_readlane(first_q, seq), k0 = __builtin_amdgcn_readlane(first_k, seq);
        t.seq_start = __builtin_amdgcn_readlane(s.start, seq); t.seq_len = __builtin_amdgcn_readlane(s.len, seq); t.seq_id = seq;
        for (int i = threadIdx.x; i < nq; i += blockDim.x) { t.origin = (nq - 1 - i) * kBlockQ; p.q_tiles[q0 + i] = t; }
        if (p.k_turns) {
          // The group's sequences, by rank, and where the first one's tiles begin (an empty sequence is in none).
          const int mine = __builtin_amdgcn_readlane(rank, seq), group = mine / turns * turns;
          int tiles[kMostTurns], start = k0;
#pragma unroll
          for (int j = 0; j < kMostTurns; j++) {
            const uint64_t at = __ballot(nk > 0 && j < turns && rank == group + j);
            tiles[j] = at ? __builtin_amdgcn_readlane(nk, __builtin_ctzll(at)) : 0;
            if (j == 0 && at) start = __builtin_amdgcn_readlane(first_k, __builtin_ctzll(at));
          }
          for (int i = threadIdx.x; i < n; i += blockDim.x) {
            int place = start + (mine - group);
#pragma unroll
            for (int j = 0; j < kMostTurns; j++) place += max(0, tiles[j] - (n - i));
            t.origin = i * p.key_tile;
            p.k_tiles[place] = t;
            p.k_turns[place] = Turn{k0, mine};
          }
        } else {
          for (int i = threadIdx.x; i < n; i += blockDim.x) { t.origin = i * p.key_tile; p.k_tiles[k0 + i] = t; }
        }
        if (threadIdx.x == 0) p.carry_base[seq] = t.carry_base;
        t.carry_base += carry_slots(nq);
      }
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
