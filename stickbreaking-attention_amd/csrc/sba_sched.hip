// cu_seqlens -> tile scheduler.
//
// The reference pads every sequence to the longest one: its grid is (num_seqs, H/2, max_len/64 + 1) programs,
// most of which exit idle on a ragged batch (stickbreaking_attention/sb_varlen/sb_varlen_fwd.py:475-479, :294).
// Here a single small kernel reads cu_seqlens on the device (no host synchronisation) and enumerates exactly the
// tiles that exist, so the one launch that follows fills the chip without padding.  Order: sequences longest
// first, and inside a sequence the heaviest tile first (the last query tile / the first key tile).  The tiles of
// one (head, sequence) are therefore resident together and sweep the same K/V (or Q/dO) rows a step or two apart,
// which keeps those rows in the XCD's L2 instead of re-fetching them from HBM, and the launch still ends with
// the cheap tiles of the short sequences.  It also lays out the per-(row, 32-key sub-tile) carries per sequence.
#include "sba_device.hpp"
#include "sba_params.hpp"
#include "sba_sched.hpp"

namespace sba {

constexpr int kBins = 4096;          // sequence length classes (query tiles per sequence, saturating)
constexpr int kSchedThreads = 1024;

constexpr int kSchedWaves = kSchedThreads / 64;

// What the waves in front of this one, and all of them, hold of `n` values per thread; upto[i]: in, a value, out, its sum over the wave's lanes up
// to this one.  `parts` must not be in use; one barrier.
template <int kN, typename V>
__device__ __forceinline__ void block_sums(V (&upto)[kN], V (&before)[kN], V (&all)[kN], V (*parts)[kSchedWaves]) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int i = 0; i < kN; i++) {
    upto[i] = sum_up_to_lane(upto[i]);
    if (lane == 63) parts[i][wave] = upto[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kN; i++) {
    const V of_waves = sum_up_to_lane(lane < kSchedWaves ? parts[i][lane] : (V)0);
    before[i] = wave > 0 ? read_lane(of_waves, wave - 1) : (V)0;
    all[i] = read_lane(of_waves, kSchedWaves - 1);
  }
}

// What bounds it is the length of its chain of steps (one workgroup): sums are formed by scans over the lanes and one exchange between the waves, and
// what all lanes of a wave add to one counter the wave adds up first.  (Training calls with one
// sequence of 4096 tokens, all others of up to 64, us, with sums over LDS, ten barriers each, and a counter for every lane / now: 2049 sequences 29.5 / 14.5;
// 600 16.9 / 8.3; 100 10.5 / 6.8.)
__global__ __launch_bounds__(kSchedThreads) void sched_kernel(SchedParams p) {
  if (blockIdx.x > 0) {      // helper workgroups: clear the region the launch was asked to clear
    const int64_t n16 = p.zero_bytes / 16, per = (n16 + gridDim.x - 2) / (gridDim.x - 1);
    const int64_t a = per * (blockIdx.x - 1), b = a + per < n16 ? a + per : n16;
    u32x4* z = reinterpret_cast<u32x4*>(p.zero_fill);
    for (int64_t i = a + threadIdx.x; i < b; i += kSchedThreads) z[i] = u32x4{0u, 0u, 0u, 0u};
    return;
  }
  __shared__ int bins[3][kBins];      // query tiles, key tiles and (row tiles) sequences of a length class, then where each class begins
  int (&qbins)[kBins] = bins[0], (&kbins)[kBins] = bins[1], (&sbins)[kBins] = bins[2];
  __shared__ uint64_t parts[2][1][kSchedWaves];
  __shared__ int bin_parts[3][kSchedWaves];
  __shared__ unsigned long long row_run, work[2];      // work: of the sequences of one row tile, and of more
  __shared__ int status, longest;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwaves = kSchedWaves;
  for (int i = threadIdx.x; i < kBins; i += kSchedThreads) { qbins[i] = 0; kbins[i] = 0; sbins[i] = 0; }
  if (threadIdx.x == 0) { row_run = 0; work[0] = work[1] = 0; longest = 0; status = kSchedOk; }
  __syncthreads();

  // Pass 1: tiles per length class (class = number of query tiles of the sequence, saturating), and the layout of the carries: a sum over the
  // sequences in front.  Every entry of cu_seqlens is checked here; the checks are local (each end against its predecessor and the token
  // count), and together they bound the tile counts and carry slots by what the caller's buffers were sized for.  What all lanes of a wave
  // add to is added up by the wave first.
  uint64_t carry_run = 0;
  for (int s0 = 0; s0 < p.num_seqs; s0 += kSchedThreads) {
    const int s = s0 + threadIdx.x;
    int start = 0, len = 0;
    if (s < p.num_seqs && !seq_bounds(p, s, &start, &len)) status = kSchedBadCu;
    const int nq = (len + kBlockQ - 1) / kBlockQ, nk = key_tiles(p, len);
    const int cls = min(nq, kBins - 1);
    // (Most sequences of a large batch are of one class.)
    const uint64_t with_keys = __ballot(nk > 0);
    const int first_cls = __builtin_amdgcn_readfirstlane(cls);
    if (first_cls > 0 && __all(cls == first_cls)) {
      const int of_q = read_lane(sum_up_to_lane(nq), 63), of_k = read_lane(sum_up_to_lane(nk), 63);
      if (lane == 0) {
        atomicAdd(&qbins[cls], of_q);
        if (p.want_key_tiles) atomicAdd(&kbins[cls], of_k);
        if (p.k_turns) atomicAdd(&sbins[cls], __builtin_popcountll(with_keys));
      }
    } else if (nq) {
      atomicAdd(&qbins[cls], nq);
      if (p.want_key_tiles) atomicAdd(&kbins[cls], nk);
      if (nk && p.k_turns) atomicAdd(&sbins[cls], 1);
    }
    if (p.k_turns) {
      const uint64_t mine = nk ? row_work(len) : 0, of_wave[2] = {wave_sum(nk > 1 ? 0 : mine), wave_sum(nk > 1 ? mine : 0)};
      if (lane < 2 && of_wave[lane]) atomicAdd(&work[lane], (unsigned long long)of_wave[lane]);
      if (nk) atomicMax(&longest, len);
    }
    if (p.row_capacity >= 0) {
      const uint64_t blocks = wave_sum(row_blocks(len));
      if (lane == 0 && blocks) atomicAdd(&row_run, (unsigned long long)blocks);
    }
    if (p.carry_rows) {
      const uint64_t mine = slots_of(p, len, nq);
      uint64_t upto[1] = {mine}, before[1], all[1];
      block_sums(upto, before, all, parts[(s0 / kSchedThreads) & 1]);
      if (s < p.num_seqs) p.carry_base[s] = (int64_t)(carry_run + before[0] + upto[0] - mine);
      carry_run += all[0];
    }
  }
  __syncthreads();
  int verdict = status;
  if (verdict == kSchedOk && p.row_capacity >= 0 && row_run > (unsigned long long)p.row_capacity) verdict = kSchedCarryOverflow;
  if (verdict == kSchedOk && p.carry_rows && (int64_t)carry_run > p.carry_capacity) verdict = kSchedCarryOverflow;      // the caller's max_seqlen (or slot count) was too small
  if (verdict != kSchedOk) {      // uniform: nothing is scheduled, every output row is zero-filled as uncovered
    if (threadIdx.x == 0) { p.counts[kCountQ] = 0; p.counts[kCountK] = 0; p.counts[kCountStatus] = verdict; p.counts[kCountCovered] = 0; }
    if (p.want_key_tiles)
      for (int h = threadIdx.x; h < p.num_heads; h += kSchedThreads) p.head_queue[h] = 0;
    return;
  }
  // Where each class begins: sums over the classes from the heaviest down.  Thread t owns bins kBins - 1 - kPer t down to kBins - kPer (t + 1).
  {
    constexpr int kPer = kBins / kSchedThreads;
    int local[3][kPer], upto[3], before[3], all[3];
#pragma unroll
    for (int b = 0; b < 3; b++) {
      upto[b] = 0;
#pragma unroll
      for (int i = 0; i < kPer; i++) { local[b][i] = bins[b][kBins - 1 - (kPer * threadIdx.x + i)]; upto[b] += local[b][i]; }
    }
    const int mine[3] = {upto[0], upto[1], upto[2]};
    block_sums(upto, before, all, bin_parts);
#pragma unroll
    for (int b = 0; b < 3; b++) {
      int base = before[b] + upto[b] - mine[b];
#pragma unroll
      for (int i = 0; i < kPer; i++) { bins[b][kBins - 1 - (kPer * threadIdx.x + i)] = base; base += local[b][i]; }
    }
  }
  __syncthreads();
  if (p.k_turns && threadIdx.x == 0) {      // (behind the classes of more than two query tiles)
    p.counts[kCountChained] = kbins[kRowTileRows / kBlockQ];
    p.counts[kCountApart] = apart_share(work[0], work[1], row_work(longest));
  }
  __syncthreads();

  // Pass 2: each sequence takes a contiguous range of slots in its class.  A wave holds `group` sequences, one per lane; a lane
  // writes the tiles of a short sequence itself, the wave those of a long one together.  (A wave per sequence took 1.1 us of
  // dependent loads for each: 151 us for 2049 sequences.)
  constexpr int kOwnTiles = 4;
  const int group = min(64, (p.num_seqs + nwaves - 1) / nwaves);
  for (int s0 = wave * group; s0 < p.num_seqs; s0 += nwaves * group) {
    const int s = s0 + lane;
    int start = 0, len = 0, qbase = 0, kbase = 0, rank = 0;
    int64_t cbase = 0;
    const bool mine = lane < group && s < p.num_seqs;
    if (mine) {
      seq_bounds(p, s, &start, &len);
      if (p.carry_rows) cbase = p.carry_base[s];      // written above by this workgroup
    }
    const int nq = (len + kBlockQ - 1) / kBlockQ, nk = p.want_key_tiles ? key_tiles(p, len) : 0;
    const int cls = min(nq, kBins - 1);
    const int first_cls = __builtin_amdgcn_readfirstlane(cls);
    if (first_cls > 0 && __all(cls == first_cls)) {      // a place for all of them
      const int upto_q = sum_up_to_lane(nq), upto_k = sum_up_to_lane(nk);
      const uint64_t with_keys = __ballot(nk > 0);
      if (lane == 0) {
        qbase = atomicAdd(&qbins[cls], read_lane(upto_q, 63));
        if (p.want_key_tiles) kbase = atomicAdd(&kbins[cls], read_lane(upto_k, 63));
        if (p.k_turns) rank = atomicAdd(&sbins[cls], __builtin_popcountll(with_keys));
      }
      qbase = __builtin_amdgcn_readfirstlane(qbase) + upto_q - nq;
      kbase = __builtin_amdgcn_readfirstlane(kbase) + upto_k - nk;
      rank = __builtin_amdgcn_readfirstlane(rank) + __builtin_popcountll(with_keys & ((1ull << lane) - 1));
    } else {
      if (nq) qbase = atomicAdd(&qbins[cls], nq);
      if (nk) kbase = atomicAdd(&kbins[cls], nk);
      if (nk && p.k_turns) rank = atomicAdd(&sbins[cls], 1);
    }
    Tile d;
    d.seq_start = start; d.seq_len = len; d.seq_id = s; d.carry_base = cbase;
    if (nq <= kOwnTiles) {
      for (int t = 0; t < nq; t++) { d.origin = (nq - 1 - t) * kBlockQ; p.q_tiles[qbase + t] = d; }      // heaviest first: the last one
      for (int t = 0; t < nk; t++) {                                                                     // ... and the first one
        d.origin = t * p.key_tile;
        p.k_tiles[kbase + t] = d;
        if (p.k_turns) p.k_turns[kbase + t] = Turn{kbase, rank};
      }
    }
    for (uint64_t left = __ballot(nq > kOwnTiles); left; left &= left - 1) {
      const int j = __builtin_ctzll(left);
      const int nq_j = __shfl(nq, j), nk_j = __shfl(nk, j), qbase_j = __shfl(qbase, j), kbase_j = __shfl(kbase, j), rank_j = __shfl(rank, j);
      Tile e;
      e.seq_start = __shfl(start, j); e.seq_len = __shfl(len, j); e.seq_id = __shfl(s, j);
      e.carry_base = (int64_t)(uint32_t)__shfl((int)cbase, j) | (int64_t)__shfl((int)(cbase >> 32), j) << 32;
      for (int t = lane; t < nq_j; t += 64) { e.origin = (nq_j - 1 - t) * kBlockQ; p.q_tiles[qbase_j + t] = e; }
      for (int t = lane; t < nk_j; t += 64) {
        e.origin = t * p.key_tile;
        p.k_tiles[kbase_j + t] = e;
        if (p.k_turns) p.k_turns[kbase_j + t] = Turn{kbase_j, rank_j};
      }
    }
  }
  __syncthreads();
  // After the scatter, the lightest bin (work 0) ends at the total count.
  if (threadIdx.x == 0) {
    p.counts[kCountQ] = qbins[0];
    p.counts[kCountK] = p.want_key_tiles ? kbins[0] : 0;
    p.counts[kCountStatus] = kSchedOk;
    int start = 0, len = (int)p.total_tokens;      // fixed-length mode: every row belongs to a sequence
    if (p.cu != nullptr) seq_bounds(p, p.num_seqs - 1, &start, &len);
    p.counts[kCountCovered] = start + len;
  }
  if (p.want_key_tiles)
    for (int h = threadIdx.x; h < p.num_heads; h += kSchedThreads) p.head_queue[h] = 0;

}

// One workgroup schedules; `clear_wgs` more clear p.zero_fill alongside.
hipError_t launch_sched(const SchedParams& p, int clear_wgs, hipStream_t stream) {
  hipLaunchKernelGGL(sched_kernel, dim3(1 + clear_wgs), dim3(kSchedThreads), 0, stream, p);
  return hipGetLastError();
}

}  // namespace sba
