// prefill_f32_mfma.hip -- f32 prefill attention on the f32 matrix
// instructions (v_mfma_f32_32x32x2_f32: exact f32 products, f32 sums) for
// the MLA head widths (dn 128, dr 64, dv 128).
//
// Bound: f32 MFMA issue.  A 32-key x 32-row unit is 160 MFMAs of 64 clocks;
// the 40 KB of K and V it reads come from L2 at 16 B per clock and CU.
//
// Split: a block owns 32 query rows of one (b, h) -- few rows, because a
// 1000-token prompt of 16 heads then still gives 512 blocks -- and its four
// waves take every fourth 32-key tile, each with its own online softmax; the
// four partial results meet in LDS at the end.  The waves share nothing in
// the loop, so there is no barrier: each streams its K and V through its own
// two 8 KB LDS stages (32 keys x 64 floats) by direct-to-LDS DMA, the next
// chunk in flight during the 32 MFMAs of the current one.  Two blocks fit a
// CU (64 KB of LDS, 256 registers), so one wave's softmax runs under the
// other's MFMAs.
//
// Both products take their operands as they lie.  S^T = K Q^T leaves lane l
// with query row l % 32 and keys 8 a + 4 (l / 32) + b in register 4 a + b;
// that register is already the B operand (row l % 32, k = l / 32) of
// O^T += V^T P^T for the key pair (8 a + b, 8 a + 4 + b), and the running
// maximum, sum and rescaling are per-lane values.
//
// 16 heads x 1000 tokens, causal: 65.6 us (78 TFLOP/s of f32 products, 50% of
// the f32 matrix peak) against 4138 us with the VALU kernel of prefill.hip;
// 16 heads x 24 tokens 10.9 against 194 us.  Relative error against 64 bits
// 2.0e-7 (VALU kernel 3.4e-7).  One 64-dim score chain per K chunk: 62.4 us,
// but more error than the VALU kernel on short prompts (1.4e-7, 1.3e-7).

#include "mfma_pipe.hpp"

namespace qmla {

namespace {

using namespace pipe;

constexpr int kRows = 32;             // query rows per block
constexpr int kKeys = 32;             // keys per tile
constexpr int kWaves = 4;
constexpr int kChunkBytes = kKeys * 64 * 4;  // 64 floats of each key
constexpr int kRingBytes = 2 * kChunkBytes;  // per wave
constexpr int kDn = 128, kDr = 64, kDv = 128;
constexpr int kChunks = (kDn + kDr + kDv) / 64;  // per tile: 2 nope, 1 rope, 2 v

// Block order.  With at most two blocks per CU all of them start at once and
// block i shares a CU with block i + CUs: the second half goes out lightest
// first, so a long row tile is paired with a short one.  More blocks than
// that go out per (b, h), heaviest tile first, (b, h) pairs dealt to the XCDs
// (block i runs on XCD i % 8), so that an XCD's L2 holds the K and V of the
// pairs in flight.
enum { kOrderPaired = 0, kOrderXcd = 1, kOrderPlain = 2 };

__device__ __forceinline__ void block_tile(int order, int tiles, int bhs, int &tile, int &bh) {
  const int i = blockIdx.x;
  if (order == kOrderXcd) {
    const int j = i >> 3;
    bh = (j / tiles) * 8 + (i & 7);
    tile = tiles - 1 - j % tiles;
    return;
  }
  const int rank = i / bhs;
  bh = i - rank * bhs;
  tile = tiles - 1 - rank;
  const int half = (tiles + 1) / 2;
  if (order == kOrderPaired && rank >= half) tile = rank - half;
}

// Starts the DMA of one 8 KB chunk: 32 rows (from sbase, `ld` bytes apart, no
// row past rmax) x 256 bytes.  Row r's 16-byte piece p lands at piece
// p ^ swz(r) of its 256 bytes; instruction t carries rows 4 t .. 4 t + 3.
// K chunks swizzle by the row (the 16 rows a quarter-wave reads at one piece
// fall on different banks); V chunks swap the two 128-byte halves of rows
// with bit 2 set (the two keys of an MFMA step differ in it).
template <bool V>
__device__ __forceinline__ void dma_chunk(const uint8_t *sbase, int ld, int rmax, int lane_in, uint32_t lds) {
  const int lane = vfresh(lane_in);  // no per-lane offsets kept across the loop
  const int sub = lane >> 4, pos = lane & 15;
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const int row = 4 * t + sub;
    const int piece = V ? pos ^ ((t & 1) << 3) : pos ^ (row & 15);
    dma16(sbase, (uint32_t)(min(row, rmax) * ld + piece * 16), lds + t * 1024);
  }
}

__global__ __launch_bounds__(kWaves * 64, 2) void k_prefill_f32_mfma(
    const float *__restrict__ q_nope, const float *__restrict__ q_rope, const float *__restrict__ k,
    const float *__restrict__ k_rope, const float *__restrict__ v, qmla_prefill_dims d, float scale,
    int causal, int order, int tiles, float *__restrict__ out) {
  __shared__ __align__(1024) uint8_t ring[kWaves * kRingBytes];
  __shared__ float stat_m[kWaves][kRows], stat_l[kWaves][kRows];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, col = lane & 31;
  int tile, bh;
  block_tile(order, tiles, d.batch * d.heads, tile, bh);
  const int b = bh / d.heads, h = bh - b * d.heads;
  const int64_t bkr = d.k_rope_heads == 1 ? b : (int64_t)b * d.k_rope_heads + h;
  const int q0 = tile * kRows;

  // one past the last key any row of the block sees
  const int last_row = min(q0 + kRows, d.seq_q) - 1;
  const int kend = causal ? min(d.seq_k, last_row + d.q_offset + 1) : d.seq_k;
  const int ktiles = (kend + kKeys - 1) / kKeys;
  const int row_abs = causal ? d.q_offset + q0 + col : kend;  // last visible key (kend: all)

  const uint8_t *kb = reinterpret_cast<const uint8_t *>(k + (int64_t)bh * d.seq_k * kDn);
  const uint8_t *rb = reinterpret_cast<const uint8_t *>(k_rope + bkr * d.seq_k * kDr);
  const uint8_t *vb = reinterpret_cast<const uint8_t *>(v + (int64_t)bh * d.seq_k * kDv);
  const uint32_t lds0 = lds_u32((const lds_char *)ring) + wave * kRingBytes;

  auto issue = [&](int kt, int c, uint32_t lds) {
    const int k0 = kt * kKeys;
    const int rmax = kend - 1 - k0;
    if (c < 2) dma_chunk<false>(kb + (int64_t)k0 * (kDn * 4) + c * 256, kDn * 4, rmax, lane, lds);
    else if (c == 2) dma_chunk<false>(rb + (int64_t)k0 * (kDr * 4), kDr * 4, rmax, lane, lds);
    else dma_chunk<true>(vb + (int64_t)k0 * (kDv * 4) + (c - 3) * 256, kDv * 4, rmax, lane, lds);
  };
  if (wave < ktiles) issue(wave, 0, lds0);

  // Q: the lane's half of its row, 4 floats of every 8 (rows past seq_q are
  // clamped; their results are not stored)
  floatx4_t q[(kDn + kDr) / 8];
  {
    const int64_t qr = (int64_t)bh * d.seq_q + min(q0 + col, d.seq_q - 1);
#pragma unroll
    for (int j = 0; j < kDn / 8; ++j)
      q[j] = *reinterpret_cast<const floatx4_t *>(q_nope + qr * kDn + 8 * j + 4 * half);
#pragma unroll
    for (int j = 0; j < kDr / 8; ++j)
      q[kDn / 8 + j] = *reinterpret_cast<const floatx4_t *>(q_rope + qr * kDr + 8 * j + 4 * half);
  }
  floatx16_t o[kDv / 32];
#pragma unroll
  for (int n = 0; n < kDv / 32; ++n)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[n][i] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  // per-lane read offsets inside a chunk
  const uint32_t kread = col * 256 + ((half ^ (col & 15)) << 4);  // piece 2 j + half: ^ 32 j
  const uint32_t vread = half * 1024 + col * 4;                   // + 128 (n ^ half)
  uint8_t *my = ring + wave * kRingBytes;

  int stage = 0;
  for (int kt = wave; kt < ktiles; kt += kWaves) {
    floatx16_t s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      // This chunk has landed; the other stage's reads have returned, so
      // the next chunk may overwrite it.
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      const uint32_t next = lds0 + (stage ^ kChunkBytes);
      if (c + 1 < kChunks) issue(kt, c + 1, next);
      else if (kt + kWaves < ktiles) issue(kt + kWaves, 0, next);
      uint8_t *base = my + stage;
      if (c < (kDn + kDr) / 64) {
        // a sum of its own per 32 dims: short chains round less than one long one
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          floatx16_t t;
#pragma unroll
          for (int i = 0; i < 16; ++i) t[i] = 0.f;
#pragma unroll
          for (int j = 4 * g; j < 4 * g + 4; ++j) {
            const floatx4_t a = *reinterpret_cast<const floatx4_t *>(base + (kread ^ (32 * j)));
#pragma unroll
            for (int i = 0; i < 4; ++i)
              t = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], q[c * 8 + j][i], t, 0, 0, 0);
          }
          s += t;
        }
      } else {
        if (c == (kDn + kDr) / 64) {
          // online softmax of the tile's scores: s becomes P^T
          const int key0 = kt * kKeys + 4 * half;
          float mx = -INFINITY;
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int key = key0 + 8 * (i >> 2) + (i & 3);
            s[i] = key < kend && key <= row_abs ? s[i] * scale : -INFINITY;
            mx = fmaxf(mx, s[i]);
          }
          mx = fmaxf(m_run, xor32_max(mx));
          const float ref = mx == -INFINITY ? 0.f : mx;  // nothing visible yet: every p is 0
          const float alpha = expf(m_run - ref);
          float sum = 0.f;
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            s[i] = expf(s[i] - ref);
            sum += s[i];
          }
          l_run = l_run * alpha + sum;
          // unchanged maxima leave O as it is (NaN compares unequal and rescales)
          if (__any(!(mx == m_run))) {
#pragma unroll
            for (int n = 0; n < kDv / 32; ++n)
#pragma unroll
              for (int i = 0; i < 16; ++i) o[n][i] *= alpha;
          }
          m_run = mx;
        }
        // value rows past kend are zeroed: 0 * V is 0 whatever the re-loaded key holds
        if (kend - kt * kKeys < kKeys)
          for (int i = (kend - kt * kKeys) * 16 + lane; i < kKeys * 16; i += 64)
            reinterpret_cast<floatx4_t *>(base)[i] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 16; ++i) {
#pragma unroll
          for (int n = 0; n < 2; ++n) {
            const float a = *reinterpret_cast<const float *>(
                base + vread + (8 * (i >> 2) + (i & 3)) * 256 + ((n ^ half) << 7));
            const int on = (c - (kDn + kDr) / 64) * 2 + n;
            o[on] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, s[i], o[on], 0, 0, 0);
          }
        }
      }
      stage ^= kChunkBytes;
    }
  }

  // Merge of the four waves: the row's common maximum and sum, then each
  // wave's weighted O^T as [row][128] through its own (idle) ring, summed in
  // wave order.  Row r's piece p sits at piece p ^ r.
  l_run = xor32_sum(l_run);
  if (half == 0) {
    stat_m[wave][col] = m_run;
    stat_l[wave][col] = l_run;
  }
  __syncthreads();
  float mx = -INFINITY;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) mx = fmaxf(mx, stat_m[w][col]);
  const float ref = mx == -INFINITY ? 0.f : mx;
  const float wt = expf(m_run - ref);
  {
    uint8_t *dst = ring + wave * kRingBytes + col * 512;
#pragma unroll
    for (int n = 0; n < kDv / 32; ++n)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const int piece = 8 * n + 2 * a + half;
        floatx4_t x = {o[n][4 * a] * wt, o[n][4 * a + 1] * wt, o[n][4 * a + 2] * wt, o[n][4 * a + 3] * wt};
        *reinterpret_cast<floatx4_t *>(dst + ((piece ^ col) << 4)) = x;
      }
  }
  __syncthreads();
  float *ob = out + ((int64_t)bh * d.seq_q + q0) * kDv;
#pragma unroll
  for (int it = 0; it < kRows / 8; ++it) {
    const int row = it * 8 + (threadIdx.x >> 5), piece = threadIdx.x & 31;
    if (q0 + row >= d.seq_q) continue;
    float rm = -INFINITY, l = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) rm = fmaxf(rm, stat_m[w][row]);
    const float rref = rm == -INFINITY ? 0.f : rm;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) l += expf(stat_m[w][row] - rref) * stat_l[w][row];
    floatx4_t x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
      x += *reinterpret_cast<const floatx4_t *>(ring + w * kRingBytes + row * 512 + ((piece ^ row) << 4));
    const float inv = l > 0.f ? 1.f / l : 0.f;
    *reinterpret_cast<floatx4_t *>(ob + (int64_t)row * kDv + piece * 4) = x * inv;
  }
}

}  // namespace

// The f32 MFMA kernel takes the MLA widths with 16-byte aligned tensors (its
// rows move in 16-byte pieces); every other call keeps the VALU kernel.
bool prefill_f32_mfma_supported(const qmla_prefill_dims &d, const float *q_nope, const float *q_rope,
                                const float *k, const float *k_rope, const float *v, const float *out) {
  const uintptr_t any = (uintptr_t)q_nope | (uintptr_t)q_rope | (uintptr_t)k | (uintptr_t)k_rope |
                        (uintptr_t)v | (uintptr_t)out;
  const int64_t blocks = (int64_t)((d.seq_q + kRows - 1) / kRows) * d.batch * d.heads;
  return d.qk_nope == kDn && d.qk_rope == kDr && d.v_dim == kDv && (any & 15) == 0 &&
         blocks < (int64_t)1 << 31 && d.seq_k <= (1 << 30) && d.seq_q <= (1 << 30) && d.q_offset <= (1 << 30);
}

qmla_status launch_prefill_f32_mfma(const qmla_prefill_dims &d, const float *q_nope, const float *q_rope,
                                    const float *k, const float *k_rope, const float *v, float scale,
                                    int causal, float *out, hipStream_t stream) {
  const int tiles = (d.seq_q + kRows - 1) / kRows;
  const int bhs = d.batch * d.heads;
  int cus = device_cu_count();
  if (cus <= 0) cus = 256;
  const int order = (int64_t)tiles * bhs <= 2 * (int64_t)cus ? kOrderPaired
                    : bhs % 8 == 0                          ? kOrderXcd
                                                            : kOrderPlain;
  k_prefill_f32_mfma<<<dim3(tiles * bhs), dim3(kWaves * 64), 0, stream>>>(
      q_nope, q_rope, k, k_rope, v, d, scale, causal, order, tiles, out);
  QMLA_LAUNCH_CHECK("k_prefill_f32_mfma");
  return QMLA_OK;
}

}  // namespace qmla
