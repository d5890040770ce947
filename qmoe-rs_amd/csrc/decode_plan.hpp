// decode_plan.hpp -- the split plan the MFMA decode kernels (decode_mfma.hip,
// decode_f32_mfma.hip) compute in the kernel itself.
#pragma once

#include "internal.hpp"

namespace qmla {
namespace {

// Sequences are cut at multiples of kPlanTok tokens: the tokens of a tile.
constexpr int kPlanTok = 32;

// ---- in-kernel split plan.  The concatenated tokens of the batch are cut
// into gridDim.x pieces of `chunk` tokens; piece i covers [i*chunk,
// (i+1)*chunk).  Each sequence is preceded by seg_tokens virtual tokens in
// this stream: a segment costs a fixed setup (Q load, prologue, partial
// store) on top of its tiles, and a piece that starts a new sequence gets
// correspondingly fewer real tokens.  A (piece, sequence) overlap of real
// tokens is a segment; every segment
// writes a partial result to its own slot: sequence b owns slots
// sb[b] .. sb[b] + ns[b] - 1 (ns[b] = pieces it touches), in piece order.
// Each block derives its own segments (no separate planning launch): the
// length prefix sums are rebuilt in the idle stage ring, and up to kSegCap
// segment descriptors are kept in LDS; a block with more segments plans
// again when its list runs out.  The block whose piece holds a sequence's
// first token (blockIdx.y == 0) records {sb, ns} for the merge.
constexpr int kSegCap = 64;

struct SegDesc {
  int32_t seq, t0, t1, slot;
};

// Exclusive scan of a[0..n) in LDS; returns the total.  Up to 512 values
// are scanned by wave 0 alone (lane-local runs, then a shuffle scan: one
// barrier in all); longer arrays by all NT threads (log-step, two barriers
// per step).
// The piece of this block.  Blocks are dealt to the 8 XCDs round-robin, so
// block i maps to piece (i % 8) * (grid / 8) + i / 8: consecutive pieces,
// i.e. the pieces of one sequence, sit on one XCD and its query rows come
// from that XCD's L2 after the first load (16-head decode 41.0-41.4 ->
// 40.5-40.8 us per step in a same-box A/B; the 128-head decode within noise).
__device__ __forceinline__ int decode_piece() {
  const int g = gridDim.x, b = blockIdx.x;
  return (g & 7) ? b : (b & 7) * (g >> 3) + (b >> 3);
}

template <int NT>
__device__ int32_t lds_exscan(int32_t *a, int32_t n, int32_t *tmp) {
  if (n <= 512) {
    if (threadIdx.x < 64) {
      const int lane = threadIdx.x;
      const int per = (n + 63) / 64;
      const int lo = min(n, lane * per), hi = min(n, lo + per);
      int32_t local = 0;
      for (int i = lo; i < hi; ++i) local += a[i];
      int32_t incl = local;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int32_t v = __shfl_up(incl, off);
        if (lane >= off) incl += v;
      }
      int32_t run = incl - local;
      for (int i = lo; i < hi; ++i) {
        const int32_t v = a[i];
        a[i] = run;
        run += v;
      }
      if (lane == 63) tmp[0] = incl;
    }
    __syncthreads();
    return tmp[0];
  }
  const int tid = threadIdx.x;
  const int per = (n + NT - 1) / NT;
  const int lo = min(n, tid * per), hi = min(n, lo + per);
  int32_t local = 0;
  for (int i = lo; i < hi; ++i) local += a[i];
  tmp[tid] = local;
  __syncthreads();
  for (int off = 1; off < NT; off <<= 1) {
    const int32_t v = tid >= off ? tmp[tid - off] : 0;
    __syncthreads();
    tmp[tid] += v;
    __syncthreads();
  }
  int32_t run = tid > 0 ? tmp[tid - 1] : 0;
  const int32_t total = tmp[NT - 1];
  for (int i = lo; i < hi; ++i) {
    const int32_t v = a[i];
    a[i] = run;
    run += v;
  }
  __syncthreads();
  return total;
}

// One planning round: fills list[0..count) with this block's segments of
// sequences >= from, sets *next to the first sequence not listed (batch
// when done).  scratch: 2 * (batch + 1) + NT int32 of idle LDS.  In the
// virtual stream, sequence b occupies [P[b], P[b + 1]) with its real
// tokens at [v0, v0 + L) = [P[b] + seg_tokens, P[b + 1]).  Sequences are
// cut only at tile boundaries (multiples of kPlanTok from the sequence start):
// the tile starting at virtual position v belongs to the piece holding v,
// so every segment starts at a multiple of kPlanTok and each of its tiles lies
// in one cache page.  A piece is at least kPlanTok long, so the pieces holding
// a sequence's tile starts are consecutive and each gets a non-empty segment.
template <int NT>
__device__ void plan_round(const int32_t *__restrict__ lens, int32_t pending, int32_t batch,
                           int32_t from, int32_t seg_tokens, int32_t *scratch, SegDesc *list,
                           int32_t *meta, int2 *__restrict__ seq_info) {
  const int tid = threadIdx.x;
  const int blocks = gridDim.x, piece = decode_piece();
  int32_t *P = scratch, *SB = scratch + batch + 1, *tmp = SB + batch + 1;
  for (int b = tid; b < batch; b += NT) P[b] = lens[b] + pending + seg_tokens;
  __syncthreads();
  const int32_t N = lds_exscan<NT>(P, batch, tmp);
  if (tid == 0) P[batch] = N;
  const int32_t chunk = max(kPlanTok, (N + blocks - 1) / blocks);
  __syncthreads();
  // pieces holding the tile starts of a sequence with real tokens [v0, v0 + L)
  auto touched = [&](int32_t v0, int32_t L) {
    return L > 0 ? (v0 + (L - 1) / kPlanTok * kPlanTok) / chunk - v0 / chunk + 1 : 0;
  };
  // sequence-relative cut at virtual position x: the first tile start >= x
  auto cut = [&](int32_t x, int32_t v0, int32_t L) {
    return x <= v0 ? 0 : min(L, (x - v0 + kPlanTok - 1) / kPlanTok * kPlanTok);
  };
  for (int b = tid; b < batch; b += NT) {
    const int32_t v0 = P[b] + seg_tokens;
    SB[b] = touched(v0, P[b + 1] - v0);
  }
  __syncthreads();
  (void)lds_exscan<NT>(SB, batch, tmp);
  if (from == 0 && blockIdx.y == 0) {
    for (int b = tid; b < batch; b += NT) {
      const int32_t v0 = P[b] + seg_tokens;
      if (min(v0 / chunk, blocks - 1) == piece)
        seq_info[b] = make_int2(SB[b], touched(v0, P[b + 1] - v0));
    }
  }
  if (tid == 0) {
    const int32_t start = min(piece * chunk, N), end = min(start + chunk, N);
    // first sequence >= from whose tokens reach past start
    int32_t lo = from, hi = batch;
    while (lo < hi) {
      const int32_t mid = (lo + hi) >> 1;
      if (P[mid + 1] > start) hi = mid; else lo = mid + 1;
    }
    int32_t cnt = 0, b = lo;
    for (; b < batch && P[b] + seg_tokens < end && cnt < kSegCap; ++b) {
      const int32_t v0 = P[b] + seg_tokens, L = P[b + 1] - v0;
      const int32_t t0 = cut(start, v0, L), t1 = cut(end, v0, L);
      if (t1 <= t0) continue;  // empty sequence, or no tile start inside the piece
      list[cnt++] = SegDesc{b, t0, t1, SB[b] + (piece - v0 / chunk)};
    }
    meta[0] = cnt;
    meta[1] = (b < batch && P[b] + seg_tokens < end) ? b : batch;
  }
  __syncthreads();
}

// The same plan for batch <= 64, computed by every wave in registers (lane b
// = sequence b): two shuffle scans and a ballot instead of LDS round trips
// and barriers, so the first tiles are requested sooner.  A piece then holds
// at most 64 <= kSegCap segments: one round.  Segment i is the i-th set bit
// of mask, in ascending sequence order as in plan_round.
struct WavePlan {
  uint64_t mask;
  int32_t t0, t1, slot;  // this lane's sequence
};

__device__ __forceinline__ int32_t wave_incl_scan(int32_t x) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int32_t v = __shfl_up(x, off);
    if (lane >= off) x += v;
  }
  return x;
}

__device__ WavePlan plan_wave(const int32_t *__restrict__ lens, int32_t pending, int32_t batch,
                              int32_t seg_tokens, int2 *__restrict__ seq_info) {
  static_assert(kSegCap >= 64, "one round per piece");
  const int lane = threadIdx.x & 63;
  const int blocks = gridDim.x, piece = decode_piece();
  const bool live = lane < batch;
  const int32_t x = live ? lens[lane] + pending + seg_tokens : 0;
  const int32_t incl = wave_incl_scan(x);  // P[b + 1]
  const int32_t N = __shfl(incl, 63);
  const int32_t chunk = max(kPlanTok, (N + blocks - 1) / blocks);
  const int32_t v0 = incl - x + seg_tokens, L = x - seg_tokens;
  const int32_t first = v0 / chunk;
  const int32_t touched = live && L > 0 ? (v0 + (L - 1) / kPlanTok * kPlanTok) / chunk - first + 1 : 0;
  const int32_t sb = wave_incl_scan(touched) - touched;
  if (blockIdx.y == 0 && (threadIdx.x >> 6) == 0 && live && min(first, blocks - 1) == piece)
    seq_info[lane] = make_int2(sb, touched);
  const int32_t start = min(piece * chunk, N), end = min(start + chunk, N);
  auto cut = [&](int32_t c) { return c <= v0 ? 0 : min(L, (c - v0 + kPlanTok - 1) / kPlanTok * kPlanTok); };
  WavePlan w;
  w.t0 = cut(start);
  w.t1 = cut(end);
  w.slot = sb + (piece - first);
  w.mask = __ballot(live && incl > start && v0 < end && w.t1 > w.t0);
  return w;
}

// One planning round of a block: the segment count; next_seq = the first
// sequence of the next round (batch when there is none).
template <int NT>
__device__ __forceinline__ int32_t plan_segments(const int32_t *__restrict__ lens, int32_t pending,
                                                 int32_t batch, int32_t &next_seq,
                                                 int32_t seg_tokens, int32_t *scratch,
                                                 SegDesc *list, int32_t *meta,
                                                 int2 *__restrict__ seq_info, WavePlan &wp) {
  if (batch <= 64) {
    wp = plan_wave(lens, pending, batch, seg_tokens, seq_info);
    next_seq = batch;
    return __builtin_popcountll(wp.mask);
  }
  plan_round<NT>(lens, pending, batch, next_seq, seg_tokens, scratch, list, meta, seq_info);
  next_seq = __builtin_amdgcn_readfirstlane(meta[1]);
  return __builtin_amdgcn_readfirstlane(meta[0]);
}

// Segment si of the round (called for si = 0, 1, ... in order).
__device__ __forceinline__ SegDesc plan_segment(int32_t si, int32_t batch, const SegDesc *list,
                                                WavePlan &wp) {
  SegDesc sg;
  if (batch <= 64) {
    const int ln = __builtin_ctzll(wp.mask);
    wp.mask &= wp.mask - 1;
    sg.seq = ln;
    sg.t0 = __builtin_amdgcn_readlane(wp.t0, ln);
    sg.t1 = __builtin_amdgcn_readlane(wp.t1, ln);
    sg.slot = __builtin_amdgcn_readlane(wp.slot, ln);
  } else {
    const SegDesc d = list[si];
    sg.seq = __builtin_amdgcn_readfirstlane(d.seq);
    sg.t0 = __builtin_amdgcn_readfirstlane(d.t0);
    sg.t1 = __builtin_amdgcn_readfirstlane(d.t1);
    sg.slot = __builtin_amdgcn_readfirstlane(d.slot);
  }
  return sg;
}

}  // namespace
}  // namespace qmla
