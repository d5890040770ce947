// decode_f32_mfma.hip -- f32 absorbed decode on the f32 matrix instructions
// (v_mfma_f32_16x16x4_f32: exact f32 products, f32 sums) for kv_lora_rank
// 512 and rope 64.
//
// Bound: for a few users' contexts, the latency chain of a block's first tile
// (lengths, first rows from HBM, merge launch) and then its tiles one after the
// other: a 32-token tile is 72 KB and 4,350 clocks of MFMA per SIMD (two waves of
// 68 MFMAs of 32 clocks), 17 B per clock and CU.  A lone block takes 3.6 us a
// tile, half of it MFMA; with 256 blocks 5.2 us, 3.6 TB/s.
//
// Split: one block of eight waves per piece of the concatenated tokens
// (decode_plan.hpp) and 16 query rows.  Waves 0-3 take the first 16 tokens of
// each 32-token tile, waves 4-7 the others.  Wave w of a group owns c_kv
// columns 128 w .. 128 w + 127 and rope columns 16 w .. 16 w + 15: the same
// slice of a row serves its share of the score's dims and its share of the
// output columns, so no wave reads another's tile data and each streams its
// slice (16 tokens x 576 B) through its own two LDS stages by direct-to-LDS
// DMA.  The waves meet once per tile, to add the four partial scores through
// LDS; the two groups keep their own online softmax and meet at the end of a
// segment.
//
// S^T = K Q^T leaves lane l with query row l % 16 and tokens 4 (l / 16) + i in
// register i, which is already the B operand of O^T += V^T P^T for the four
// tokens i, 4 + i, 8 + i, 12 + i.
//
// 8 users of 300-4000 tokens, 16 heads (20.5K tokens, 47 MB): 26 us, decode
// and merge, 1.8 TB/s, against 304 us with the VALU kernel of decode.hip, which
// reads the cache once per query row; 8 x 4000 tokens 32 us, 2.3 TB/s.  Relative
// error against 64 bits 3.1e-7 to 3.3e-7 (VALU kernel 5.2e-7 to 5.6e-7).

#include "decode_plan.hpp"
#include "mfma_pipe.hpp"

namespace qmla {

namespace {

using namespace pipe;

constexpr int kR = 512, kDr = 64, kRowBytes = (kR + kDr) * 4;
constexpr int kRowsPerBlock = 16;
constexpr int kThreads = 512;
constexpr int kHalfTok = kPlanTok / 2;             // tokens of a group per tile
constexpr int kSliceKv = 128 * 4, kSliceRope = 16 * 4;  // a wave's bytes per token
constexpr int kStage = kHalfTok * (kSliceKv + kSliceRope);
constexpr int kRing = 8 * 2 * kStage;
constexpr int kExch = 8 * 1024;                    // partial scores: [wave][lane] x 16 B
constexpr int kStats = 16 * 2 * 4;                 // group 1's maximum and sum per row
constexpr size_t kLds = kRing + kExch + kStats + kSegCap * sizeof(SegDesc) + 16;
static_assert(kLds <= 160 * 1024, "LDS budget");

// 4-byte aligned vectors: queries, outputs and workspace need no more.
typedef float floatx4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint16_t u16x4_a2 __attribute__((ext_vector_type(4), aligned(2)));

template <typename QT>
__device__ __forceinline__ floatx4_t load_q4(const QT *p) {
  if constexpr (sizeof(QT) == 4) {
    return *reinterpret_cast<const floatx4_a4 *>(p);
  } else {
    const u16x4_a2 u = *reinterpret_cast<const u16x4_a2 *>(p);
    return floatx4_t{bf16_bits_to_f32(u[0]), bf16_bits_to_f32(u[1]), bf16_bits_to_f32(u[2]),
                     bf16_bits_to_f32(u[3])};
  }
}

// DMA of this wave's slice of 16 tokens at `rows` (the slice's first c_kv
// byte of token 0; `rope` likewise); tokens past `last` re-load that token.
// c_kv: instruction t carries tokens 2 t, 2 t + 1, 512 B each; token r's
// 16-byte piece p lands at piece p ^ r, so that the 16 tokens of a score
// operand and the 4 x 64 B of a V^T operand fall on different banks.  rope:
// one instruction, token r's piece p at p ^ (r / 4).
__device__ __forceinline__ void dma_slice(const uint8_t *rows, const uint8_t *rope, int last, int lane_in,
                                          uint32_t lds) {
  const int lane = vfresh(lane_in);
#pragma unroll
  for (int t = 0; t < kHalfTok / 2; ++t) {
    const int r = 2 * t + (lane >> 5), pos = lane & 31;
    dma16(rows, (uint32_t)(min(r, last) * kRowBytes + ((pos ^ r) << 4)), lds + t * 1024);
  }
  const int r = lane >> 2, pos = lane & 3;
  dma16(rope, (uint32_t)(min(r, last) * kRowBytes + ((pos ^ (r >> 2)) << 4)), lds + kHalfTok * kSliceKv);
}

// Block barrier that waits for this wave's LDS traffic only: the DMA of the
// next tile stays in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Reduction over the four lanes of a query row (l, l ^ 16, l ^ 32, l ^ 48).
__device__ __forceinline__ float row_max(float x) {
  x = fmaxf(x, __shfl_xor(x, 16));
  return xor32_max(x);
}
__device__ __forceinline__ float row_sum(float x) {
  x += __shfl_xor(x, 16);
  return xor32_sum(x);
}

template <typename QT>
__global__ __launch_bounds__(kThreads, 1) void k_decode_f32_mfma(
    const uint64_t *__restrict__ pages, int32_t pt_width, int32_t pt_shift, const int32_t *__restrict__ lens,
    int32_t batch, const QT *__restrict__ q_lat, const QT *__restrict__ q_rope, int32_t rows, float scale,
    int32_t pending, int2 *__restrict__ seq_info, float *__restrict__ part_o, float *__restrict__ part_lse) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  float *exch = reinterpret_cast<float *>(lds + kRing);
  float *stats = reinterpret_cast<float *>(lds + kRing + kExch);
  SegDesc *seg_list = reinterpret_cast<SegDesc *>(lds + kRing + kExch + kStats);
  int32_t *seg_meta = reinterpret_cast<int32_t *>(seg_list + kSegCap);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w = wave & 3, group = wave >> 2;
  const int col = lane & 15, quad = lane >> 4;
  const int row = blockIdx.y * kRowsPerBlock + col;  // this lane's query row
  const int row_c = min(row, rows - 1);              // rows past the last are not stored
  const uint8_t *my = lds + wave * 2 * kStage;
  const uint32_t my_u = lds_u32((const lds_char *)lds) + wave * 2 * kStage;

  // operand offsets inside a stage: score operand piece 4 j + quad of token
  // col (^ 64 j), its rope piece, and V^T of tokens 4 quad + i (^ 64 cb)
  const uint32_t k_off = col * kSliceKv + ((quad ^ col) << 4);
  const uint32_t r_off = kHalfTok * kSliceKv + col * kSliceRope + ((quad ^ (col >> 2)) << 4);
  uint32_t v_off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    v_off[i] = (4 * quad + i) * kSliceKv + (quad << 6) + (((col >> 2) ^ i) << 4) + ((col & 3) << 2);

  int32_t next_seq = 0;
  do {
    WavePlan wp;
    const int32_t nseg = plan_segments<kThreads>(lens, pending, batch, next_seq, kDecodeF32SegTokens,
                                                 reinterpret_cast<int32_t *>(lds), seg_list, seg_meta, seq_info, wp);
    for (int32_t si = 0; si < nseg; ++si) {
      const SegDesc sg = plan_segment(si, batch, seg_list, wp);
      const uint64_t *prow = pages + (int64_t)sg.seq * pt_width;
      const int T = sg.t1 - sg.t0;
      const int ntiles = (T + kPlanTok - 1) / kPlanTok;
      // A tile starts at a multiple of kPlanTok tokens, so it lies in one
      // page.  A group whose 16 tokens all lie past the end re-loads the
      // segment's last one and masks it.
      auto issue = [&](int it) {
        const int t = sg.t0 + it * kPlanTok;
        const int first = min(group * kHalfTok, T - 1 - it * kPlanTok);
        const uint8_t *base = reinterpret_cast<const uint8_t *>(prow[t >> pt_shift]) +
                              (int64_t)((t & ((1 << pt_shift) - 1)) + first) * kRowBytes;
        dma_slice(base + w * kSliceKv, base + kR * 4 + w * kSliceRope, T - 1 - it * kPlanTok - first, lane,
                  my_u + (it & 1) * kStage);
      };
      issue(0);

      floatx4_t q[9];  // 16 j + 4 quad of the wave's c_kv dims, then its rope dims
      const int64_t qrow = (int64_t)sg.seq * rows + row_c;
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = load_q4(q_lat + qrow * kR + 128 * w + 16 * j + 4 * quad);
      q[8] = load_q4(q_rope + qrow * kDr + 16 * w + 4 * quad);

      floatx4_t o[8];
#pragma unroll
      for (int n = 0; n < 8; ++n) o[n] = floatx4_t{0.f, 0.f, 0.f, 0.f};
      float m_run = -INFINITY, l_run = 0.f;
      for (int it = 0; it < ntiles; ++it) {
        // this tile's slice has landed, and every read of the other stage
        // (and of the exchanged scores) has returned
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        if (it + 1 < ntiles) issue(it + 1);
        const uint8_t *st = my + (it & 1) * kStage;
        // partial scores, in three short sums
        floatx4_t s[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          s[c] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int j = 3 * c; j < 3 * c + 3; ++j) {
            const floatx4_t a = *reinterpret_cast<const floatx4_t *>(st + (j < 8 ? k_off ^ (64 * j) : r_off));
#pragma unroll
            for (int i = 0; i < 4; ++i)
              s[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], q[j][i], s[c], 0, 0, 0);
          }
        }
        lds_barrier();  // the exchange of the last tile has been read
        *reinterpret_cast<floatx4_t *>(exch + (wave * 64 + lane) * 4) = (s[0] + s[1]) + s[2];
        lds_barrier();
        floatx4_t p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 4; ++k) p += *reinterpret_cast<const floatx4_t *>(exch + ((group * 4 + k) * 64 + lane) * 4);
        const int valid = T - it * kPlanTok - group * kHalfTok - 4 * quad;  // tokens of this lane
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          p[i] = i < valid ? p[i] * scale : -INFINITY;
          mx = fmaxf(mx, p[i]);
        }
        mx = fmaxf(m_run, row_max(mx));
        const float ref = mx == -INFINITY ? 0.f : mx;  // nothing valid yet: every p is 0
        const float alpha = expf(m_run - ref);
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          p[i] = expf(p[i] - ref);
          sum += p[i];
        }
        l_run = l_run * alpha + sum;
        // unchanged maxima leave O as it is (NaN compares unequal and rescales)
        if (__any(!(mx == m_run))) {
#pragma unroll
          for (int n = 0; n < 8; ++n) o[n] *= alpha;
        }
        m_run = mx;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int n = 0; n < 8; ++n) {
            const float a = *reinterpret_cast<const float *>(st + (v_off[i] ^ (64 * n)));
            o[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, p[i], o[n], 0, 0, 0);
          }
      }

      // The two groups' results: group 1 leaves its statistics and O^T in
      // LDS, group 0 (same lanes, same rows and columns) adds and stores.
      l_run = row_sum(l_run);
      floatx4_t *dump = reinterpret_cast<floatx4_t *>(lds + (4 + w) * 2 * kStage) + lane;
      if (group == 1) {
#pragma unroll
        for (int n = 0; n < 8; ++n) dump[64 * n] = o[n];
        if (w == 0 && quad == 0) {
          stats[col] = m_run;
          stats[16 + col] = l_run;
        }
      }
      __syncthreads();
      if (group == 0) {
        const float m1 = stats[col], l1 = stats[16 + col];
        const float mx = fmaxf(m_run, m1);
        const float ref = mx == -INFINITY ? 0.f : mx;
        const float a0 = expf(m_run - ref), a1 = expf(m1 - ref);
        const float l = l_run * a0 + l1 * a1;
        const float inv = 1.f / l;
        const int64_t prow_o = (int64_t)sg.slot * rows + row;
        if (row < rows) {
#pragma unroll
          for (int n = 0; n < 8; ++n)
            *reinterpret_cast<floatx4_a4 *>(part_o + prow_o * kR + 128 * w + 16 * n + 4 * quad) =
                (o[n] * a0 + dump[64 * n] * a1) * inv;
          if (w == 0 && quad == 0) part_lse[prow_o] = mx + logf(l);
        }
      }
      __syncthreads();  // the dump is read: the next segment may overwrite it
    }
  } while (next_seq < batch);
}

// Log-sum-exp merge of the partial slots: a block per (sequence, query row,
// 256 columns), wave k taking slots k, k + 8, ... with four loads in flight;
// the eight partial sums are added through LDS in wave order.  Empty
// sequences get zeros and lse = -inf.
__global__ __launch_bounds__(512) void k_decode_merge_f32(int32_t rows, const int2 *__restrict__ seq_info,
                                                          const float *__restrict__ part_o,
                                                          const float *__restrict__ part_lse,
                                                          float *__restrict__ out, float *__restrict__ out_lse,
                                                          int32_t *__restrict__ adv_lens, int32_t adv) {
  __shared__ floatx4_t acc_s[8][64];
  const int b = blockIdx.x, m = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int2 info = seq_info[b];
  const int n = info.y;
  // lengths grow by the pending tokens the decode attended (it has finished)
  if (adv_lens && m == 0 && blockIdx.z == 0 && threadIdx.x == 0) adv_lens[b] += adv;
  const int64_t qrow = (int64_t)b * rows + m;
  const float *lse = part_lse + (int64_t)info.x * rows + m;
  float mx = -INFINITY, wsum = 0.f;
  for (int k = lane; k < n; k += 64) mx = fmaxf(mx, lse[(int64_t)k * rows]);
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) mx = fmaxf(mx, __shfl_xor(mx, d));
  for (int k = lane; k < n; k += 64) wsum += expf(lse[(int64_t)k * rows] - mx);
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) wsum += __shfl_xor(wsum, d);
  const int c = blockIdx.z * 256 + lane * 4;
  const float *src = part_o + ((int64_t)info.x * rows + m) * kR + c;
  floatx4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = wave; k < n; k += 8) {
    const floatx4_t x = *reinterpret_cast<const floatx4_a4 *>(src + (int64_t)k * rows * kR);
    acc += x * expf(lse[(int64_t)k * rows] - mx);
  }
  acc_s[wave][lane] = acc;
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int k = 1; k < 8; ++k) acc += acc_s[k][lane];
  if (n > 0) acc *= 1.f / wsum;
  *reinterpret_cast<floatx4_a4 *>(out + qrow * kR + c) = acc;
  if (out_lse && lane == 0 && blockIdx.z == 0) out_lse[qrow] = n > 0 ? mx + logf(wsum) : -INFINITY;
}

}  // namespace

bool decode_f32_mfma_supported(int32_t r, int32_t dr) { return r == kR && dr == kDr; }

qmla_status launch_decode_f32_mfma(const DecodeArgs &a, hipStream_t stream) {
  // the merge's grid has a row per query row
  QMLA_REQUIRE(a.rows <= 65535, QMLA_ERR_SHAPE, "rows %d > 65535", a.rows);
  const dim3 grid(a.blocks, (a.rows + kRowsPerBlock - 1) / kRowsPerBlock);
  const PageTable tab = a.cache->table();
  if (a.q_dtype == QMLA_BF16) {
    auto k = k_decode_f32_mfma<uint16_t>;
    QMLA_TRY(ensure_dynamic_lds((const void *)k, kLds));
    k<<<grid, dim3(kThreads), kLds, stream>>>(tab.pages, tab.width, tab.shift, a.cache->d_lens, a.batch,
                                              (const uint16_t *)a.q_lat, (const uint16_t *)a.q_rope, a.rows, a.scale,
                                              a.pending, a.seq_info, a.part_o, a.part_lse);
  } else {
    auto k = k_decode_f32_mfma<float>;
    QMLA_TRY(ensure_dynamic_lds((const void *)k, kLds));
    k<<<grid, dim3(kThreads), kLds, stream>>>(tab.pages, tab.width, tab.shift, a.cache->d_lens, a.batch,
                                              (const float *)a.q_lat, (const float *)a.q_rope, a.rows, a.scale,
                                              a.pending, a.seq_info, a.part_o, a.part_lse);
  }
  QMLA_LAUNCH_CHECK("k_decode_f32_mfma");
  k_decode_merge_f32<<<dim3(a.batch, a.rows, kR / 256), dim3(512), 0, stream>>>(
      a.rows, a.seq_info, a.part_o, a.part_lse, a.out, a.out_lse, a.advance ? a.cache->d_lens : nullptr, a.pending);
  QMLA_LAUNCH_CHECK("k_decode_merge_f32");
  return QMLA_OK;
}

}  // namespace qmla
