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

// Exclusive prefix sum over bins taken from the heaviest bin downwards; bins[] becomes the start offsets.
__device__ void descending_offsets(int* bins, int* scratch) {
  constexpr int kPer = kBins / kSchedThreads;
  const int t = threadIdx.x;
  // thread t owns bins (kBins-1 - kPer*t) down to (kBins-1 - kPer*t - kPer + 1)
  int local[kPer], sum = 0;
#pragma unroll
  for (int i = 0; i < kPer; i++) { local[i] = bins[kBins - 1 - (kPer * t + i)]; sum += local[i]; }
  scratch[t] = sum;
  __syncthreads();
  for (int d = 1; d < kSchedThreads; d <<= 1) {
    const int v = (t >= d) ? scratch[t - d] : 0;
    __syncthreads();
    scratch[t] += v;
    __syncthreads();
  }
  int base = scratch[t] - sum;
#pragma unroll
  for (int i = 0; i < kPer; i++) { bins[kBins - 1 - (kPer * t + i)] = base; base += local[i]; }
  __syncthreads();
}

__global__ __launch_bounds__(kSchedThreads) void sched_kernel(SchedParams p) {
  if (blockIdx.x > 0) {      // helper workgroups: clear the region the launch was asked to clear
    const int64_t n16 = p.zero_bytes / 16, per = (n16 + gridDim.x - 2) / (gridDim.x - 1);
    const int64_t a = per * (blockIdx.x - 1), b = a + per < n16 ? a + per : n16;
    u32x4* z = reinterpret_cast<u32x4*>(p.zero_fill);
    for (int64_t i = a + threadIdx.x; i < b; i += kSchedThreads) z[i] = u32x4{0u, 0u, 0u, 0u};
    return;
  }
  __shared__ int qbins[kBins];
  __shared__ int kbins[kBins];
  __shared__ int sbins[kBins];      // row tiles: sequences per length class
  __shared__ int scratch[kSchedThreads];
  __shared__ long long carry_run;
  __shared__ unsigned long long row_run, work[2];      // work: of the sequences of one row tile, and of more
  __shared__ int status, longest;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwaves = kSchedThreads / 64;
  for (int i = threadIdx.x; i < kBins; i += kSchedThreads) { qbins[i] = 0; kbins[i] = 0; sbins[i] = 0; }
  if (threadIdx.x == 0) { carry_run = 0; row_run = 0; work[0] = work[1] = 0; longest = 0; status = kSchedOk; }
  __syncthreads();

  // Pass 1: tiles per length class (class = number of query tiles of the sequence, saturating).  Every entry of
  // cu_seqlens is checked here; the checks are local (each end against its predecessor and the token count), and
  // together they bound the tile counts and carry slots by what the caller's buffers were sized for.
  for (int s = threadIdx.x; s < p.num_seqs; s += kSchedThreads) {
    int start, len;
    if (!seq_bounds(p, s, &start, &len)) status = kSchedBadCu;
    const int nq = (len + kBlockQ - 1) / kBlockQ, nk = (len + p.key_tile - 1) / p.key_tile;
    const int cls = min(nq, kBins - 1);
    if (nq) atomicAdd(&qbins[cls], nq);
    if (nk && p.want_key_tiles) atomicAdd(&kbins[cls], nk);
    if (nk && p.k_turns) {
      atomicAdd(&sbins[cls], 1);
      atomicAdd(&work[nk > 1], (unsigned long long)row_work(len));
      atomicMax(&longest, len);
    }
    if (p.row_capacity >= 0 && row_blocks(len) > 0) atomicAdd(&row_run, (unsigned long long)row_blocks(len));
  }
  __syncthreads();
  if (threadIdx.x == 0 && status == kSchedOk && p.row_capacity >= 0 && row_run > (unsigned long long)p.row_capacity) status = kSchedCarryOverflow;
  __syncthreads();
  if (status != kSchedOk) {      // uniform: nothing is scheduled, every output row is zero-filled as uncovered
    if (threadIdx.x == 0) { p.counts[kCountQ] = 0; p.counts[kCountK] = 0; p.counts[kCountStatus] = status; p.counts[kCountCovered] = 0; }
    if (p.want_key_tiles)
      for (int h = threadIdx.x; h < p.num_heads; h += kSchedThreads) p.head_queue[h] = 0;
    return;
  }
  descending_offsets(qbins, scratch);
  if (p.want_key_tiles) descending_offsets(kbins, scratch);
  if (p.k_turns) descending_offsets(sbins, scratch);
  if (p.k_turns && threadIdx.x == 0) {      // (behind the classes of more than two query tiles)
    p.counts[kCountChained] = kbins[kRowTileRows / kBlockQ];
    p.counts[kCountApart] = apart_share(work[0], work[1], row_work(longest));
  }

  // Carry layout: exclusive prefix sum of carry_slots(M_s) over sequences (block-wide, chunked).
  if (p.want_carry_base) {
    for (int s0 = 0; s0 < p.num_seqs; s0 += kSchedThreads) {
      const int s = s0 + threadIdx.x;
      int start = 0, len = 0;
      if (s < p.num_seqs) seq_bounds(p, s, &start, &len);
      const long long mine = carry_slots((len + kBlockQ - 1) / kBlockQ);
      // inclusive scan of `mine` through 64-bit shuffles would need two passes; sequences per chunk are
      // few enough for a shared-memory Hillis-Steele scan on the low/high words kept as long long.
      __shared__ long long sc[kSchedThreads];
      sc[threadIdx.x] = mine;
      __syncthreads();
      for (int d = 1; d < kSchedThreads; d <<= 1) {
        const long long v = (threadIdx.x >= d) ? sc[threadIdx.x - d] : 0;
        __syncthreads();
        sc[threadIdx.x] += v;
        __syncthreads();
      }
      const long long base = carry_run;
      if (s < p.num_seqs) p.carry_base[s] = base + sc[threadIdx.x] - mine;
      __syncthreads();
      if (threadIdx.x == kSchedThreads - 1) carry_run = base + sc[threadIdx.x];
      __syncthreads();
    }
    if (carry_run > p.carry_capacity) {      // uniform: the caller's max_seqlen (or slot count) was too small
      if (threadIdx.x == 0) { p.counts[kCountQ] = 0; p.counts[kCountK] = 0; p.counts[kCountStatus] = kSchedCarryOverflow; p.counts[kCountCovered] = 0; }
      if (p.want_key_tiles)
        for (int h = threadIdx.x; h < p.num_heads; h += kSchedThreads) p.head_queue[h] = 0;
      return;
    }
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
      if (p.want_carry_base) cbase = p.carry_base[s];      // written above by this workgroup
    }
    const int nq = (len + kBlockQ - 1) / kBlockQ, nk = p.want_key_tiles ? (len + p.key_tile - 1) / p.key_tile : 0;
    const int cls = min(nq, kBins - 1);
    if (nq) qbase = atomicAdd(&qbins[cls], nq);
    if (nk) kbase = atomicAdd(&kbins[cls], nk);
    if (nk && p.k_turns) rank = atomicAdd(&sbins[cls], 1);
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
