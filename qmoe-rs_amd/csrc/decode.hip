// decode.hip -- absorbed-latent MLA decode: work plan, f32 core, merge and
// the C entry points.
//
// Replaces the attention core of MlaAttention::forward_with_cache
// (src/model.rs:294-303: scores over the decompressed per-head cache,
// softmax, times V) by the absorbed form over the shared latent cache:
//   s_t = scale * (q_lat . c_t + q_rope . kpe_t),  o_lat = sum_t p_t c_t
// (the W_UK absorption into q_lat and the W_UV product on o_lat happen in
// the layer; see layer.hip).
//
// Work split: the tokens of all sequences, concatenated, are cut into
// `blocks` equal pieces (one or a few per compute unit); every (piece,
// sequence) overlap is a segment.  A sequence covered by one segment is
// written straight to the output; otherwise each segment writes a partial
// (o / l, log-sum-exp) slot and k_decode_merge combines them.

#include <algorithm>
#include <atomic>
#include <cmath>
#include <mutex>

#include "internal.hpp"

namespace qmla {

namespace {

constexpr int kPlanThreads = 1024;

// Exclusive scan of n ints held in LDS (in place); returns the total.
// Every thread of the block must call it.
__device__ int32_t block_exclusive_scan(int32_t *a, int32_t n, int32_t *tmp) {
  const int tid = threadIdx.x;
  const int per = (n + kPlanThreads - 1) / kPlanThreads;
  const int lo = min(n, tid * per), hi = min(n, lo + per);
  int32_t local = 0;
  for (int i = lo; i < hi; ++i) local += a[i];
  tmp[tid] = local;
  __syncthreads();
  // Hillis-Steele over the kPlanThreads partial sums.
  for (int off = 1; off < kPlanThreads; off <<= 1) {
    int32_t v = tid >= off ? tmp[tid - off] : 0;
    __syncthreads();
    tmp[tid] += v;
    __syncthreads();
  }
  int32_t run = tid > 0 ? tmp[tid - 1] : 0;
  const int32_t total = tmp[kPlanThreads - 1];
  for (int i = lo; i < hi; ++i) {
    int32_t v = a[i];
    a[i] = run;
    run += v;
  }
  __syncthreads();
  return total;
}

// One block builds the segment list.  LDS: P[batch] prefix, S[batch] slot
// base, C[blocks] segment counts, tmp[kPlanThreads].
__global__ __launch_bounds__(kPlanThreads) void k_decode_plan(const int32_t *__restrict__ lens,
                                                              int32_t pending, int32_t batch,
                                                              int32_t blocks, int32_t chunk,
                                                              DecodePlanView plan) {
  extern __shared__ int32_t sm[];
  int32_t *P = sm;               // [batch + 1]
  int32_t *S = P + batch + 1;    // [batch]
  int32_t *C = S + batch;        // [blocks + 1]
  int32_t *tmp = C + blocks + 1; // [kPlanThreads]
  const int tid = threadIdx.x;

  for (int b = tid; b < batch; b += kPlanThreads) P[b] = lens[b] + pending;
  __syncthreads();
  const int32_t N = block_exclusive_scan(P, batch, tmp);
  if (tid == 0) P[batch] = N;
  __syncthreads();

  // slots per sequence
  for (int b = tid; b < batch; b += kPlanThreads) {
    int32_t T = P[b + 1] - P[b];
    int32_t n = 0;
    if (T > 0) {
      int32_t first = min(P[b] / chunk, blocks - 1);
      int32_t last = min((P[b] + T - 1) / chunk, blocks - 1);
      n = last - first + 1;
    }
    S[b] = n;
    plan.seq_nslots[b] = n;
  }
  __syncthreads();
  (void)block_exclusive_scan(S, batch, tmp);
  for (int b = tid; b < batch; b += kPlanThreads) plan.seq_slot_base[b] = S[b];

  // segments per piece: sequences overlapping [start, end)
  for (int i = tid; i < blocks; i += kPlanThreads) {
    int32_t start = min(i * chunk, N);
    int32_t end = (i == blocks - 1) ? N : min((i + 1) * chunk, N);
    int32_t cnt = 0;
    if (start < end) {
      // first sequence whose end P[b+1] > start
      int32_t lo = 0, hi = batch - 1;
      while (lo < hi) {
        int32_t mid = (lo + hi) >> 1;
        if (P[mid + 1] > start) hi = mid; else lo = mid + 1;
      }
      for (int32_t b = lo; b < batch && P[b] < end; ++b)
        if (P[b + 1] > P[b]) ++cnt;
    }
    C[i] = cnt;
  }
  __syncthreads();
  const int32_t total_segs = block_exclusive_scan(C, blocks, tmp);
  for (int i = tid; i < blocks; i += kPlanThreads) plan.seg_start[i] = C[i];
  if (tid == 0) plan.seg_start[blocks] = total_segs;

  for (int i = tid; i < blocks; i += kPlanThreads) {
    int32_t start = min(i * chunk, N);
    int32_t end = (i == blocks - 1) ? N : min((i + 1) * chunk, N);
    if (start >= end) continue;
    int32_t lo = 0, hi = batch - 1;
    while (lo < hi) {
      int32_t mid = (lo + hi) >> 1;
      if (P[mid + 1] > start) hi = mid; else lo = mid + 1;
    }
    int32_t out = C[i];
    for (int32_t b = lo; b < batch && P[b] < end; ++b) {
      int32_t T = P[b + 1] - P[b];
      if (T <= 0) continue;
      int32_t first = min(P[b] / chunk, blocks - 1);
      int32_t nsl = plan.seq_nslots[b];
      DecodeSegment sg;
      sg.seq = b;
      sg.t0 = max(start, P[b]) - P[b];
      sg.t1 = min(end, P[b + 1]) - P[b];
      sg.slot = nsl == 1 ? -1 : S[b] + (i - first);
      plan.segs[out++] = sg;
    }
  }
}

// ---------------------------------------------------------------- f32 core
// One block per (piece, query row).  Per 64-token chunk: 4 threads per
// token form the 576-wide dot product, the chunk's scores update an online
// softmax, and each thread accumulates up to kColsPerThread latent columns.
constexpr int kF32Threads = 256;
constexpr int kF32Tok = 64;
constexpr int kColsPerThread = 4;  // r <= 1024

template <typename QT>
__device__ inline float load_q(const QT *p, int64_t i) {
  if constexpr (sizeof(QT) == 4) return p[i];
  else return bf16_bits_to_f32(p[i]);
}

template <typename QT>
__global__ __launch_bounds__(kF32Threads) void k_decode_f32(
    PageTable tab, const QT *__restrict__ q_lat, const QT *__restrict__ q_rope, int32_t rows, int32_t r,
    int32_t dr, float scale, DecodePlanView plan, float *__restrict__ out,
    float *__restrict__ out_lse, float *__restrict__ part_o, float *__restrict__ part_lse) {
  extern __shared__ float qs[];  // [r + dr]
  __shared__ float sc[kF32Tok];
  const int tid = threadIdx.x;
  const int piece = blockIdx.x;
  const int m = blockIdx.y;
  const int w = r + dr;
  const int32_t s0 = plan.seg_start[piece], s1 = plan.seg_start[piece + 1];
  for (int32_t si = s0; si < s1; ++si) {
    const DecodeSegment sg = plan.segs[si];
    const int64_t qrow = (int64_t)sg.seq * rows + m;
    __syncthreads();
    for (int c = tid; c < r; c += kF32Threads) qs[c] = load_q(q_lat, qrow * r + c);
    for (int c = tid; c < dr; c += kF32Threads) qs[r + c] = load_q(q_rope, qrow * dr + c);
    __syncthreads();
    // token t of the segment: row sg.t0 + t of the sequence, via its pages
    auto row_at = [&](int32_t t) {
      return reinterpret_cast<const float *>(tab.row(sg.seq, (int64_t)sg.t0 + t, (int64_t)w * 4));
    };
    const int32_t T = sg.t1 - sg.t0;
    float m_run = -INFINITY, l_run = 0.f;
    float acc[kColsPerThread];
#pragma unroll
    for (int k = 0; k < kColsPerThread; ++k) acc[k] = 0.f;
    for (int32_t t0 = 0; t0 < T; t0 += kF32Tok) {
      const int tt = tid >> 2, part = tid & 3;
      float d = 0.f;
      if (t0 + tt < T) {
        const float *row = row_at(t0 + tt);
        for (int c = part; c < w; c += 4) d += qs[c] * row[c];
      }
      d += __shfl_xor(d, 1);
      d += __shfl_xor(d, 2);
      if (part == 0) sc[tt] = (t0 + tt < T) ? d * scale : -INFINITY;
      __syncthreads();
      float cmax = -INFINITY;
      for (int j = 0; j < kF32Tok; ++j) cmax = fmaxf(cmax, sc[j]);
      const float m_new = fmaxf(m_run, cmax);
      const float alpha = (m_run == -INFINITY) ? 0.f : expf(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int k = 0; k < kColsPerThread; ++k) acc[k] *= alpha;
      const int nt = min(kF32Tok, T - t0);
      for (int j = 0; j < nt; ++j) {
        const float p = expf(sc[j] - m_new);
        l_run += p;
        const float *row = row_at(t0 + j);
#pragma unroll
        for (int k = 0; k < kColsPerThread; ++k) {
          const int c = tid + k * kF32Threads;
          if (c < r) acc[k] += p * row[c];
        }
      }
      m_run = m_new;
      __syncthreads();
    }
    const float inv = 1.f / l_run;
    const float lse = m_run + logf(l_run);
    if (sg.slot < 0) {
#pragma unroll
      for (int k = 0; k < kColsPerThread; ++k) {
        const int c = tid + k * kF32Threads;
        if (c < r) out[qrow * r + c] = acc[k] * inv;
      }
      if (out_lse && tid == 0) out_lse[qrow] = lse;
    } else {
      const int64_t prow = (int64_t)sg.slot * rows + m;
#pragma unroll
      for (int k = 0; k < kColsPerThread; ++k) {
        const int c = tid + k * kF32Threads;
        if (c < r) part_o[prow * r + c] = acc[k] * inv;
      }
      if (tid == 0) part_lse[prow] = lse;
    }
  }
}

// One block per (sequence, query row): log-sum-exp merge of the partial
// slots; empty sequences get zeros and lse = -inf.
__global__ __launch_bounds__(256) void k_decode_merge(int32_t rows, int32_t r, DecodePlanView plan,
                                                       const float *__restrict__ part_o,
                                                       const float *__restrict__ part_lse,
                                                       float *__restrict__ out,
                                                       float *__restrict__ out_lse,
                                                       int32_t *__restrict__ adv_lens, int32_t adv) {
  const int b = blockIdx.x, m = blockIdx.y, tid = threadIdx.x;
  // lengths grow by the pending tokens the decode attended (it has finished)
  if (adv_lens && m == 0 && tid == 0) adv_lens[b] += adv;
  const int32_t n = plan.seq_nslots[b];
  const int64_t qrow = (int64_t)b * rows + m;
  if (n == 1) return;
  if (n == 0) {
    for (int c = tid; c < r; c += blockDim.x) out[qrow * r + c] = 0.f;
    if (out_lse && tid == 0) out_lse[qrow] = -INFINITY;
    return;
  }
  const int32_t base = plan.seq_slot_base[b];
  float mx = -INFINITY;
  for (int k = 0; k < n; ++k) mx = fmaxf(mx, part_lse[(int64_t)(base + k) * rows + m]);
  float wsum = 0.f;
  for (int k = 0; k < n; ++k) wsum += expf(part_lse[(int64_t)(base + k) * rows + m] - mx);
  const float inv = 1.f / wsum;
  for (int c = tid; c < r; c += blockDim.x) {
    float a = 0.f;
    for (int k = 0; k < n; ++k) {
      const int64_t prow = (int64_t)(base + k) * rows + m;
      a += expf(part_lse[prow] - mx) * part_o[prow * r + c];
    }
    out[qrow * r + c] = a * inv;
  }
  if (out_lse && tid == 0) out_lse[qrow] = mx + logf(wsum);
}

inline size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

}  // namespace

DecodeWorkspace decode_workspace_layout(int32_t batch, int32_t rows, int32_t r, int32_t blocks,
                                        bool mfma) {
  DecodeWorkspace w;
  w.slots = blocks + batch;
  size_t plan = mfma ? sizeof(int2) * (size_t)batch
                     : sizeof(int32_t) * (blocks + 1) +
                           sizeof(DecodeSegment) * (size_t)(blocks + batch) +
                           2 * sizeof(int32_t) * batch;
  const size_t prow = mfma ? (size_t)((rows + 31) / 32) * 32 : (size_t)rows;
  w.plan_bytes = align256(plan);
  w.part_o_off = w.plan_bytes;
  // partial outputs: f32, or bf16 on the MFMA path (its log-sum-exp stays f32)
  const size_t pelt = mfma ? sizeof(uint16_t) : sizeof(float);
  w.part_lse_off = w.part_o_off + align256(pelt * (size_t)w.slots * prow * r);
  w.total = w.part_lse_off + align256(sizeof(float) * (size_t)w.slots * prow);
  return w;
}

DecodePlanView decode_plan_view(void *ws, int32_t batch, int32_t blocks) {
  DecodePlanView v;
  char *p = static_cast<char *>(ws);
  v.seg_start = reinterpret_cast<int32_t *>(p);
  p += sizeof(int32_t) * (blocks + 1);
  p = reinterpret_cast<char *>((reinterpret_cast<uintptr_t>(p) + 15) & ~uintptr_t(15));
  v.segs = reinterpret_cast<DecodeSegment *>(p);
  p += sizeof(DecodeSegment) * (size_t)(blocks + batch);
  v.seq_slot_base = reinterpret_cast<int32_t *>(p);
  p += sizeof(int32_t) * batch;
  v.seq_nslots = reinterpret_cast<int32_t *>(p);
  return v;
}

qmla_status launch_decode_plan(const qmla_kv_cache *cache, int32_t pending, int32_t batch,
                               int32_t blocks, int32_t chunk, DecodePlanView plan,
                               hipStream_t stream) {
  size_t lds = sizeof(int32_t) * ((size_t)batch + 1 + batch + blocks + 1 + kPlanThreads);
  k_decode_plan<<<dim3(1), dim3(kPlanThreads), lds, stream>>>(cache->d_lens, pending, batch,
                                                             blocks, chunk, plan);
  QMLA_LAUNCH_CHECK("k_decode_plan");
  return QMLA_OK;
}

qmla_status launch_decode_merge(int32_t batch, int32_t rows, int32_t r, DecodePlanView plan,
                                const float *part_o, const float *part_lse, float *out,
                                float *out_lse, int32_t *adv_lens, int32_t adv,
                                hipStream_t stream) {
  k_decode_merge<<<dim3(batch, rows), dim3(256), 0, stream>>>(rows, r, plan, part_o, part_lse,
                                                             out, out_lse, adv_lens, adv);
  QMLA_LAUNCH_CHECK("k_decode_merge");
  return QMLA_OK;
}

qmla_status decode_shape_supported(const qmla_kv_cache *c, int32_t rows) {
  if (c->dtype == QMLA_BF16) {
    QMLA_REQUIRE(decode_mfma_supported(rows, c->r, c->dr), QMLA_ERR_UNSUPPORTED,
                 "bf16 decode for kv_lora_rank %d, rope %d", c->r, c->dr);
    QMLA_REQUIRE(rows <= 65535 * 128, QMLA_ERR_SHAPE, "too many query rows");
    return QMLA_OK;
  }
  QMLA_REQUIRE(c->r <= kF32Threads * kColsPerThread, QMLA_ERR_UNSUPPORTED,
               "kv_lora_rank %d > %d", c->r, kF32Threads * kColsPerThread);
  QMLA_REQUIRE(rows <= 65535, QMLA_ERR_SHAPE, "rows %d > 65535", rows);
  return QMLA_OK;
}

qmla_status launch_decode_f32(const DecodeArgs &a, hipStream_t stream) {
  QMLA_REQUIRE(a.r <= kF32Threads * kColsPerThread, QMLA_ERR_UNSUPPORTED,
               "kv_lora_rank %d > %d", a.r, kF32Threads * kColsPerThread);
  QMLA_REQUIRE(a.rows <= 65535, QMLA_ERR_SHAPE, "rows %d > 65535", a.rows);
  dim3 grid(a.blocks, a.rows), block(kF32Threads);
  size_t lds = sizeof(float) * (a.r + a.dr);
  const PageTable tab = a.cache->table();
  if (a.q_dtype == QMLA_F32) {
    k_decode_f32<float><<<grid, block, lds, stream>>>(
        tab, (const float *)a.q_lat, (const float *)a.q_rope, a.rows, a.r, a.dr, a.scale, a.plan,
        a.out, a.out_lse, a.part_o, a.part_lse);
  } else {
    k_decode_f32<uint16_t><<<grid, block, lds, stream>>>(
        tab, (const uint16_t *)a.q_lat, (const uint16_t *)a.q_rope, a.rows, a.r, a.dr, a.scale,
        a.plan, a.out, a.out_lse, a.part_o, a.part_lse);
  }
  QMLA_LAUNCH_CHECK("k_decode_f32");
  return QMLA_OK;
}

}  // namespace qmla

using namespace qmla;

namespace {

qmla_status validate_decode(const qmla_decode_dims *d, const qmla_kv_cache *c) {
  QMLA_REQUIRE(d && c, QMLA_ERR_INVALID_ARG, "NULL dims or cache");
  QMLA_REQUIRE(d->batch > 0 && d->batch <= c->num_seqs, QMLA_ERR_SHAPE,
               "batch %d outside [1, %d]", d->batch, c->num_seqs);
  QMLA_REQUIRE(d->batch <= kMaxPlanBatch, QMLA_ERR_UNSUPPORTED, "batch %d > %d", d->batch,
               kMaxPlanBatch);
  QMLA_REQUIRE(d->rows > 0, QMLA_ERR_SHAPE, "rows must be > 0");
  QMLA_REQUIRE(d->kv_lora_rank == c->r && d->rope_dim == c->dr, QMLA_ERR_SHAPE,
               "dims (%d, %d) differ from the cache's (%d, %d)", d->kv_lora_rank, d->rope_dim,
               c->r, c->dr);
  int64_t total = 0;
  for (int32_t i = 0; i < d->batch; ++i) total += c->h_lens[i];
  // the in-kernel plan adds decode_mfma_seg_tokens() virtual tokens per sequence
  const int64_t virt =
      total + (int64_t)d->batch * decode_mfma_seg_tokens(d->rows, d->kv_lora_rank, d->rope_dim);
  QMLA_REQUIRE(virt < (int64_t)1 << 31, QMLA_ERR_UNSUPPORTED, "%lld tokens in one call",
               (long long)total);
  return QMLA_OK;
}

// Number of pieces: enough to fill the device, but no piece shorter than a
// minimum so that per-piece overhead (q load, partial write) stays small.
// The MFMA plans count the virtual tokens they add per sequence: without them
// 16 sequences of 100 tokens made 13 pieces of 444 virtual tokens, several
// sequences to a piece.  f32: a lone block takes 3.6 us for a 32-token tile, so
// few tokens go out one tile to a piece (278 tokens 24.0 us in 3 pieces, 13.6 in
// 11; 8 x 278 27.8 in 18, 14.3 in 86), for at most 32 rows and 64 sequences: their
// partials stay below 22 MB.  Beyond, pieces of 128 tokens without the virtual
// ones are not the best (16 rows, 64 x 100 tokens 23.7 us, 65 x 100 41.8; the VALU
// kernel took 200).  bf16: two tiles (16
// heads, 128 / 64 / 32 tokens a piece: 1 x 200 14.1 / 12.5 / 12.5 us, 1 x 4097
// 15.3 / 14.8 / 17.8, 16 x 100 14.5 / 12.5 / 12.6; 128 heads, 1 x 500 21.8 /
// 19.1 / 18.8, 4 x 1000 24.0 / 23.1 / 26.0).  The VALU path keeps 128.
// The count never falls when lengths grow; workspace_bytes_auto below makes the
// workspace's size grow with rows and batch too.
// `coarse`: pieces of 128 tokens on every path, for the fixed scratch where it
// holds no more.
int32_t choose_blocks(const qmla_decode_dims *d, const qmla_kv_cache *c, int32_t requested,
                      bool coarse = false) {
  int64_t total = 0;
  for (int32_t i = 0; i < d->batch; ++i) total += c->h_lens[i];
  if (requested > 0) return std::min<int32_t>(requested, kMaxPlanBlocks);
  int cus = device_cu_count();
  if (cus <= 0) cus = 256;
  const bool bf16 = c->dtype == QMLA_BF16 && decode_mfma_supported(d->rows, d->kv_lora_rank, d->rope_dim);
  int per_cu = bf16 ? decode_mfma_blocks_per_cu(d->rows, d->kv_lora_rank, d->rope_dim)
                    : decode_f32_blocks_per_cu(d->kv_lora_rank, d->rope_dim);
  int64_t target = (int64_t)cus * per_cu;
  int64_t min_tokens = 128;
  if (bf16 && !coarse) {
    min_tokens = 64;
    total += (int64_t)d->batch * decode_mfma_seg_tokens(d->rows, d->kv_lora_rank, d->rope_dim);
  } else if (!coarse && c->dtype == QMLA_F32 && decode_f32_mfma_supported(d->kv_lora_rank, d->rope_dim) &&
             d->rows <= 32 && d->batch <= 64) {
    min_tokens = 32;
    total += (int64_t)d->batch * kDecodeF32SegTokens;
  }
  int64_t by_work = (total + min_tokens - 1) / min_tokens;
  int64_t blocks = std::max<int64_t>(1, std::min(target, by_work));
  return (int32_t)std::min<int64_t>(blocks, kMaxPlanBlocks);
}

// Pieces the bf16 plan launches of the `blocks` it may.  Above 128 rows each
// piece is a block per 128 rows, and at rank 512 a compute unit holds one block:
// no more pieces than one round takes (256 rows, 4 x 4000 tokens 50.4 -> 33.8 us,
// 64 x 1000 88 -> 64, 64 x 4000 200 -> 161).  Then pieces of two to four tiles become whole tiles, since cut at 67 tokens some hold three tiles and
// the rest two, with more partials to merge than pieces of three (16 heads, 4 x
// 4000: 18.8 -> 16.7 us).  At 33 .. 64 rows many sequences have too few slots each
// to gain (48 rows, whole tiles / as cut: 10 x 2000 24.4 / 25.4, 2 x 10000 27.5 /
// 29.0, but 16 x 1000 26.8 / 26.1, 32 x 500 27.5 / 25.5, 64 x 200 28.3 / 24.8, 100 x
// 200 34.6 / 32.8).  Above 64 rows, where a piece's partial is larger than
// the tokens of two tiles, a sequence of more than 80 pieces takes three: its
// merge is the longer part (128 heads, 8192 + 15 x 10 tokens 40.4 -> 35.7 us; with
// up to 24 pieces per sequence two stay better, 8 x 1000 25.2 us against 26.3).  One
// tile in all is one piece (1 x 16 9.04 -> 8.81 us); several are not held to their
// number, since the cuts would fall worse (4 x 100 11.2 / 12.2, 8 x 16 of rank 64
// 7.3 / 9.0).
int32_t launch_blocks(const qmla_decode_dims *d, const qmla_kv_cache *c, int32_t blocks) {
  if (d->rows > 128 && d->kv_lora_rank == 512) {
    int cus = device_cu_count();
    if (cus <= 0) cus = 256;
    blocks = std::min(blocks, std::max(1, cus / ((d->rows + 127) / 128)));
  }
  int64_t total = (int64_t)d->batch * decode_mfma_seg_tokens(d->rows, d->kv_lora_rank, d->rope_dim);
  int32_t longest = 0;
  for (int32_t i = 0; i < d->batch; ++i) {
    total += c->h_lens[i];
    longest = std::max(longest, c->h_lens[i]);
  }
  if (d->batch == 1 && longest <= 32) return 1;
  int64_t tiles = (total + 32LL * blocks - 1) / (32LL * blocks);
  if (tiles < 2 || tiles > 4) return blocks;
  if (d->rows > 32 && d->rows <= 64 && d->batch > 15) return blocks;
  if (d->rows > 64 && longest > 80 * 64) tiles = std::max<int64_t>(tiles, 3);
  return (int32_t)std::max<int64_t>(1, std::min<int64_t>(blocks, (total + 32 * tiles - 1) / (32 * tiles)));
}

// Workspace of an automatic split: what the call itself needs, or a call of
// fewer rows or sequences over the same cache, whichever is more.  The piece
// count depends on the row class (up to 32, up to 64, more) and in f32 on the
// batch (up to 64, more), and steps down where a class ends: 65 sequences x 100
// tokens of 16 rows make 51 pieces in f32, 64 of them 256.  Within a class the
// size grows with every dimension, so the largest call of each class bounds it.
size_t workspace_bytes_auto(const qmla_decode_dims *d, const qmla_kv_cache *c) {
  size_t need = 0;
  for (int32_t rows : {32, 64, d->rows})
    for (int32_t batch : {64, d->batch}) {
      const qmla_decode_dims e{std::min(batch, d->batch), std::min(rows, d->rows), d->kv_lora_rank, d->rope_dim};
      need = std::max(need, decode_workspace_layout(e.batch, e.rows, e.kv_lora_rank, choose_blocks(&e, c, 0),
                                                    c->dtype == QMLA_BF16)
                                .total);
    }
  return need;
}

qmla_status decode_impl(const qmla_decode_dims *d, const qmla_kv_cache *c, qmla_dtype q_dtype,
                        const void *q_latent, const void *q_rope, double scale, float *out,
                        float *out_lse, int32_t splits, void *ws, size_t ws_bytes,
                        qmla_stream stream) {
  QMLA_TRY(validate_decode(d, c));
  QMLA_REQUIRE(valid_dtype(q_dtype), QMLA_ERR_INVALID_ARG, "bad q dtype");
  QMLA_REQUIRE(q_latent && out, QMLA_ERR_INVALID_ARG, "NULL q_latent or out");
  QMLA_REQUIRE(q_rope || d->rope_dim == 0, QMLA_ERR_INVALID_ARG, "NULL q_rope");
  QMLA_REQUIRE(splits >= 0, QMLA_ERR_INVALID_ARG, "negative split count");
  QMLA_REQUIRE(std::isfinite(scale), QMLA_ERR_INVALID_ARG, "non-finite scale");
  return decode_launch(d, c, q_dtype, q_latent, q_rope, scale, out, out_lse, splits, ws, ws_bytes,
                       0, false, as_stream(stream));
}

}  // namespace

qmla_status qmla::decode_launch(const qmla_decode_dims *d, const qmla_kv_cache *c,
                                qmla_dtype q_dtype, const void *q_latent, const void *q_rope,
                                double scale, float *out, float *out_lse, int32_t splits, void *ws,
                                size_t ws_bytes, int32_t pending, bool advance, hipStream_t s) {
  const int32_t blocks = choose_blocks(d, c, splits);
  const bool mfma = c->dtype == QMLA_BF16;
  if (mfma)
    QMLA_REQUIRE(decode_mfma_supported(d->rows, d->kv_lora_rank, d->rope_dim),
                 QMLA_ERR_UNSUPPORTED, "bf16 decode for kv_lora_rank %d, rope %d",
                 d->kv_lora_rank, d->rope_dim);
  DecodeWorkspace lay = decode_workspace_layout(d->batch, d->rows, d->kv_lora_rank, blocks, mfma);
  QMLA_REQUIRE(ws != nullptr && ws_bytes >= lay.total, QMLA_ERR_WORKSPACE,
               "workspace of %zu bytes < required %zu", ws_bytes, lay.total);
  DecodePlanView plan{};
  const bool f32_mfma = !mfma && decode_f32_mfma_supported(d->kv_lora_rank, d->rope_dim);
  if (!mfma && !f32_mfma) {
    plan = decode_plan_view(ws, d->batch, blocks);
    int64_t total = 0;
    for (int32_t i = 0; i < d->batch; ++i) total += c->h_lens[i];
    int32_t chunk = (int32_t)std::max<int64_t>(1, (total + blocks - 1) / blocks);
    QMLA_TRY(launch_decode_plan(c, pending, d->batch, blocks, chunk, plan, s));
  }
  DecodeArgs a;
  a.cache = c;
  a.batch = d->batch;
  a.rows = d->rows;
  a.r = d->kv_lora_rank;
  a.dr = d->rope_dim;
  a.q_lat = q_latent;
  a.q_rope = q_rope;
  a.q_dtype = q_dtype;
  a.scale = (float)scale;
  a.out = out;
  a.out_lse = out_lse;
  a.plan = plan;
  a.seq_info = reinterpret_cast<int2 *>(ws);
  a.part_o = reinterpret_cast<float *>(static_cast<char *>(ws) + lay.part_o_off);
  a.part_lse = reinterpret_cast<float *>(static_cast<char *>(ws) + lay.part_lse_off);
  a.blocks = mfma && splits <= 0 ? launch_blocks(d, c, blocks) : blocks;
  a.pending = pending;
  a.advance = advance;
  if (mfma) return launch_decode_mfma(a, s);  // decode + merge
  if (f32_mfma) return launch_decode_f32_mfma(a, s);
  QMLA_TRY(launch_decode_f32(a, s));
  return launch_decode_merge(d->batch, d->rows, d->kv_lora_rank, plan, a.part_o, a.part_lse, out,
                             out_lse, advance ? c->d_lens : nullptr, pending, s);
}

namespace {

// ------------------------------------------- allocation-free decode -----
// Scratch of qmla_decode_absorbed_noalloc: the decode workspace (plan or
// per-sequence slot table, split partials and their log-sum-exp) lives in
// this file-scope device array instead of a caller buffer.  Each device the
// library runs on holds its own copy for the life of the process.  In host
// code `scratch` names a host-side stand-in, never the device copy: the
// device address comes from hipGetSymbolAddress, once per device, and only
// that pointer is handed to kernels.  Nothing in it needs clearing: every
// call writes each slot entry and partial it later reads.
constexpr size_t kNoAllocScratchBytes = QMLA_DECODE_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

constexpr int kMaxScratchDevices = 64;
std::atomic<void *> g_scratch_ptr[kMaxScratchDevices];
std::mutex g_scratch_mu;

// Device address of this device's scratch (resolved on the first call on
// the device, with it current).
qmla_status noalloc_scratch(void **out) {
  int dev = 0;
  QMLA_HIP(hipGetDevice(&dev));
  QMLA_REQUIRE(dev >= 0 && dev < kMaxScratchDevices, QMLA_ERR_UNSUPPORTED,
               "device ordinal %d >= %d", dev, kMaxScratchDevices);
  void *p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!p) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    p = g_scratch_ptr[dev].load(std::memory_order_relaxed);
    if (!p) {
      QMLA_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
      QMLA_REQUIRE(p != nullptr, QMLA_ERR_HIP, "no device address for the decode scratch");
      g_scratch_ptr[dev].store(p, std::memory_order_release);
    }
  }
  *out = p;
  return QMLA_OK;
}

}  // namespace

extern "C" {

qmla_status qmla_decode_absorbed_noalloc(const qmla_decode_dims *dims, const qmla_kv_cache *cache,
                                         qmla_dtype q_dtype, const void *q_latent,
                                         const void *q_rope, double scale, float *out_latent,
                                         float *out_lse, qmla_stream stream) {
  QMLA_TRY(validate_decode(dims, cache));
  // the pieces of the workspace entry point where the scratch holds their
  // partials, else pieces of 128 tokens
  auto need_of = [&](int32_t blocks) {
    return decode_workspace_layout(dims->batch, dims->rows, dims->kv_lora_rank, blocks,
                                   cache->dtype == QMLA_BF16)
        .total;
  };
  const int32_t coarse = choose_blocks(dims, cache, 0, /*coarse=*/true);
  const size_t need = need_of(coarse);
  QMLA_REQUIRE(need <= kNoAllocScratchBytes, QMLA_ERR_UNSUPPORTED,
               "decode needs %zu bytes of scratch; the allocation-free entry point has %zu "
               "(use qmla_decode_absorbed with a workspace)",
               need, kNoAllocScratchBytes);
  const int32_t splits = need_of(choose_blocks(dims, cache, 0)) <= kNoAllocScratchBytes ? 0 : coarse;
  void *ws = nullptr;
  QMLA_TRY(noalloc_scratch(&ws));
  return decode_impl(dims, cache, q_dtype, q_latent, q_rope, scale, out_latent, out_lse,
                     splits, ws, kNoAllocScratchBytes, stream);
}

qmla_status qmla_decode_workspace_bytes_splits(const qmla_decode_dims *dims,
                                               const qmla_kv_cache *cache, int32_t num_splits,
                                               size_t *bytes) {
  QMLA_REQUIRE(bytes, QMLA_ERR_INVALID_ARG, "bytes is NULL");
  QMLA_TRY(validate_decode(dims, cache));
  QMLA_REQUIRE(num_splits >= 0, QMLA_ERR_INVALID_ARG, "negative split count");
  if (num_splits == 0) {
    *bytes = workspace_bytes_auto(dims, cache);
    return QMLA_OK;
  }
  int32_t blocks = choose_blocks(dims, cache, num_splits);
  *bytes = decode_workspace_layout(dims->batch, dims->rows, dims->kv_lora_rank, blocks,
                                   cache->dtype == QMLA_BF16)
               .total;
  return QMLA_OK;
}

qmla_status qmla_decode_workspace_bytes(const qmla_decode_dims *dims, const qmla_kv_cache *cache,
                                        size_t *bytes) {
  return qmla_decode_workspace_bytes_splits(dims, cache, 0, bytes);
}

qmla_status qmla_decode_absorbed(const qmla_decode_dims *dims, const qmla_kv_cache *cache,
                                 qmla_dtype q_dtype, const void *q_latent, const void *q_rope,
                                 double scale, float *out_latent, float *out_lse, void *workspace,
                                 size_t workspace_bytes, qmla_stream stream) {
  return decode_impl(dims, cache, q_dtype, q_latent, q_rope, scale, out_latent, out_lse, 0,
                     workspace, workspace_bytes, stream);
}

qmla_status qmla_decode_absorbed_splits(const qmla_decode_dims *dims, const qmla_kv_cache *cache,
                                        qmla_dtype q_dtype, const void *q_latent,
                                        const void *q_rope, double scale, float *out_latent,
                                        float *out_lse, int32_t num_splits, void *workspace,
                                        size_t workspace_bytes, qmla_stream stream) {
  return decode_impl(dims, cache, q_dtype, q_latent, q_rope, scale, out_latent, out_lse,
                     num_splits, workspace, workspace_bytes, stream);
}

}  // extern "C"
