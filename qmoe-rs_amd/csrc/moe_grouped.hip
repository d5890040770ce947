// moe_grouped.hip -- the QMoE layer's expert products for calls of many
// tokens (src/moe.rs:40-130): routing and quantisation of four tokens per
// block, and a grouped GEMM over the experts' 2-bit weights.
//
// Same exact integer form as moe_packed.hip (codes times three signed 8-bit
// digits of the activation, int32 sums on v_mfma_i32_32x32x32_i8), so every
// result has the same bits as there; what differs is the tiling.  The
// decode-sized kernel quantises 10 vectors per block and spends 7 VALU
// operations per MFMA on the codes; with hundreds of tokens per expert that
// repeats both for every 10 vectors.  Here a vector is quantised once, to
// memory, and a wave's decoded codes serve 32 tokens.
//
// Digit rows.  A vector of K values becomes a row of `pitch` = 4 K bytes: per
// 32-code chunk 96 bytes [digit][half][16], in the MFMA's lane order
// (moe_packed.hip), and at byte 3 K its DigitMeta.  A row fits the f32 row it
// came from, so the hidden activations are quantised in place.

#include <cmath>

#include "mfma_pipe.hpp"
#include "moe_internal.hpp"

namespace qmla {
namespace {

using namespace pipe;

typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x16_t __attribute__((ext_vector_type(16)));

constexpr int kGroupTok = 32;        // tokens per tile
constexpr int kRouteTok = 4;         // tokens per routing block
constexpr int kRouteThreads = 1024;
constexpr int kGemmThreads = 256;
constexpr int kQuantThreads = 128;
constexpr int kGroupedMaxK = 8192;   // widths the quantisers hold in registers
constexpr int kBadExp = 0x7fffffff;  // exponent marking a vector with inf/NaN

struct DigitMeta {
  int64_t qsum;
  int32_t e;
  int32_t pad;
};

// Exponent of a vector whose largest magnitude has the bits mb: max |q| <= 2^22.
__device__ __forceinline__ int vector_exp(uint32_t mb) {
  if (mb >= 0x7f800000u) return kBadExp;
  if (mb == 0) return 0;
  int ex;
  frexpf(__uint_as_float(mb), &ex);  // max |x| < 2^ex
  return 22 - ex;
}

// Digits of 16 consecutive values (unit u = values 16 u .. 16 u + 15 of the
// vector) into the vector's digit row; returns the sum of their integers.
__device__ __forceinline__ long long quant_unit(const floatx4_t (&f)[4], int e, int u, uint8_t *row) {
  uint32_t w[3][4] = {};
  long long sq = 0;
#pragma unroll
  for (int j = 0; j < 16; ++j) {  // j = 4 b + v -> byte b of word v
    const int q = e == kBadExp ? 0 : (int)rintf(ldexpf(f[j >> 2][j & 3], e));
    const int d0 = ((q + 128) & 255) - 128;
    const int q1 = (q - d0) >> 8;
    const int d1 = ((q1 + 128) & 255) - 128;
    const int d2 = (q1 - d1) >> 8;
    const int v = j & 3, sh = 8 * (j >> 2);
    w[0][v] |= (uint32_t)(d0 & 255) << sh;
    w[1][v] |= (uint32_t)(d1 & 255) << sh;
    w[2][v] |= (uint32_t)(d2 & 255) << sh;
    sq += q;
  }
  // values 128 g + 64 h + 16 c: chunk 4 g + c, half h
  const int chunk = (u >> 3) * 4 + (u & 3), half = (u >> 2) & 1;
#pragma unroll
  for (int p = 0; p < 3; ++p)
    *reinterpret_cast<u32x4_t *>(row + chunk * 96 + p * 32 + half * 16) =
        u32x4_t{w[p][0], w[p][1], w[p][2], w[p][3]};
  return sq;
}

__device__ __forceinline__ uint32_t abs_bits(floatx4_t v) {
  const u32x4_t m = __builtin_bit_cast(u32x4_t, v) & 0x7fffffffu;
  return max(max(m[0], m[1]), max(m[2], m[3]));
}

// Gate logits, ranks, softmax weights (k_moe_route's sums and orders, four
// tokens per block) and the tokens' digit rows.  The gate rows are read once
// per four tokens: one token per block moved the whole gate weight per token.
// LDS: x [4][H], logits [4][E].
__global__ __launch_bounds__(kRouteThreads) void k_moe_route_quant(
    const float *__restrict__ xs, const float *__restrict__ gw, int T, int E, int H, int topk,
    int32_t *__restrict__ sel, float *__restrict__ selw, int32_t *__restrict__ user_idx,
    float *__restrict__ user_w, uint8_t *__restrict__ dig, uint32_t pitch) {
  extern __shared__ __attribute__((aligned(16))) float lds_x[];
  float *lg = lds_x + kRouteTok * H;
  __shared__ uint32_t vmax[kRouteTok];
  __shared__ unsigned long long vsum[kRouteTok];
  __shared__ float stat_m[kRouteTok], stat_s[kRouteTok];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int t0 = blockIdx.x * kRouteTok, nt = min(kRouteTok, T - t0);
  const int H4 = H >> 2;
  if (tid < kRouteTok) {
    vmax[tid] = 0;
    vsum[tid] = 0;
  }
  __syncthreads();
  floatx4_t *x4 = reinterpret_cast<floatx4_t *>(lds_x);
  // a token past the end repeats the last one; none of its results is stored
  for (int t = 0; t < kRouteTok; ++t) {
    const floatx4_t *src = reinterpret_cast<const floatx4_t *>(xs + (int64_t)(t0 + min(t, nt - 1)) * H);
    uint32_t m = 0;
    for (int i = tid; i < H4; i += kRouteThreads) {
      const floatx4_t v = src[i];
      x4[t * H4 + i] = v;
      m = max(m, abs_bits(v));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o));
    if (lane == 0 && m) atomicMax(&vmax[t], m);
  }
  __syncthreads();
  for (int e = wave; e < E; e += kRouteThreads / 64) {
    const floatx4_t *w = reinterpret_cast<const floatx4_t *>(gw + (int64_t)e * H);
    float s[kRouteTok] = {};
    constexpr int U = 8;
    for (int base = 0; base < H4; base += 64 * U) {
      floatx4_t a[U];
#pragma unroll
      for (int u = 0; u < U; ++u) a[u] = w[min(base + lane + 64 * u, H4 - 1)];  // branch-free loads
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = base + lane + 64 * u;
        if (i >= H4) continue;
#pragma unroll
        for (int t = 0; t < kRouteTok; ++t) {
          const floatx4_t x = x4[t * H4 + i];
          s[t] += x[0] * a[u][0] + x[1] * a[u][1] + x[2] * a[u][2] + x[3] * a[u][3];
        }
      }
    }
#pragma unroll
    for (int t = 0; t < kRouteTok; ++t) {
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) s[t] += __shfl_xor(s[t], o);
      if (lane == 0) lg[t * E + e] = s[t];
    }
  }
  // digit rows, four waves per token
  const int units = H >> 4, tq = wave & (kRouteTok - 1);
  if (tq < nt) {
    const int e = vector_exp(vmax[tq]);
    long long sq = 0;
    for (int u = (wave / kRouteTok) * 64 + lane; u < units; u += kRouteThreads / kRouteTok) {
      floatx4_t f[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) f[j] = x4[tq * H4 + 4 * u + j];
      sq += quant_unit(f, e, u, dig + (int64_t)(t0 + tq) * pitch);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sq += __shfl_xor(sq, o);
    if (lane == 0) atomicAdd(&vsum[tq], (unsigned long long)sq);
  }
  __syncthreads();
  if (tid < nt) {
    DigitMeta *meta = reinterpret_cast<DigitMeta *>(dig + (int64_t)(t0 + tid) * pitch + 3 * (int64_t)H);
    meta->qsum = (long long)vsum[tid];
    meta->e = vector_exp(vmax[tid]);
  }
  if (wave < nt) {
    const float *l = lg + wave * E;
    float mx = -INFINITY;
    for (int e = lane; e < E; e += 64) mx = fmaxf(mx, l[e]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    float se = 0.f;
    for (int e = lane; e < E; e += 64) se += expf(l[e] - mx);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) se += __shfl_xor(se, o);
    if (lane == 0) {
      stat_m[wave] = mx;
      stat_s[wave] = se;
    }
  }
  __syncthreads();
  // ranks by (logit descending, index ascending); NaN ranks as -inf
  for (int i = tid; i < nt * E; i += kRouteThreads) {
    const int t = i / E, e = i - t * E;
    const float *l = lg + t * E;
    const float v = l[e] != l[e] ? -INFINITY : l[e];
    int rank = 0;
    for (int j = 0; j < E; ++j) {
      const float u = l[j] != l[j] ? -INFINITY : l[j];
      rank += (u > v) || (u == v && j < e);
    }
    if (rank < topk) {
      const float w = expf(l[e] - stat_m[t]) / stat_s[t];
      const int64_t o = (int64_t)(t0 + t) * topk + rank;
      sel[o] = e;
      selw[o] = w;
      if (user_idx) user_idx[o] = e;
      if (user_w) user_w[o] = w;
    }
  }
}

// f32 rows [rows][K] (pitch 4 K bytes) to digit rows, in place: a block holds
// its whole row in registers before it writes.  U units of 16 per thread.
template <int U>
__global__ __launch_bounds__(kQuantThreads) void k_moe_quant(uint8_t *__restrict__ rows, int K) {
  __shared__ uint32_t vmax;
  __shared__ unsigned long long vsum;
  const int tid = threadIdx.x, lane = tid & 63, units = K >> 4;
  uint8_t *row = rows + (int64_t)blockIdx.x * K * 4;
  if (tid == 0) {
    vmax = 0;
    vsum = 0;
  }
  __syncthreads();
  floatx4_t f[U][4];
  uint32_t m = 0;
#pragma unroll
  for (int i = 0; i < U; ++i) {
    const int u = tid + kQuantThreads * i;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
      if (u < units) f[i][j] = reinterpret_cast<const floatx4_t *>(row)[4 * u + j];
      m = max(m, abs_bits(f[i][j]));
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o));
  if (lane == 0) atomicMax(&vmax, m);
  __syncthreads();  // also: every value of the row has been read
  const int e = vector_exp(vmax);
  long long sq = 0;
#pragma unroll
  for (int i = 0; i < U; ++i) {
    const int u = tid + kQuantThreads * i;
    if (u < units) sq += quant_unit(f[i], e, u, row);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sq += __shfl_xor(sq, o);
  if (lane == 0) atomicAdd(&vsum, (unsigned long long)sq);
  __syncthreads();
  if (tid == 0) {
    DigitMeta *meta = reinterpret_cast<DigitMeta *>(row + 3 * (int64_t)K);
    meta->qsum = (long long)vsum;
    meta->e = e;
  }
}

struct GroupedArgs {
  const uint8_t *w[2];   // packed [experts][M][K / 4]
  const float *scale[2];  // [experts][M]
  int64_t w_stride;      // bytes per expert
  int64_t s_stride;      // scales per expert
  int32_t M, K;
  const uint8_t *dig;    // digit rows, `pitch` bytes apart
  uint32_t pitch;
  int32_t src_div;       // digit row of slot s = s / src_div
  const int4 *tiles;     // {expert, first bin position, tokens, -}
  const int32_t *ntiles;
  const int32_t *slots;  // bin position -> slot
  int32_t row_blocks;
  float *out;            // out[slot * ld_out + row]
  int64_t ld_out;
};

__device__ __forceinline__ i32x4_t decode_codes(uint32_t w) {
  return i32x4_t{(int)(w & 0x03030303u), (int)((w >> 2) & 0x03030303u), (int)((w >> 4) & 0x03030303u),
                 (int)((w >> 6) & 0x03030303u)};
}

// One tile of 32 tokens of one expert by 4 waves.  A wave owns four 32-row
// code operands (NMAT = 2: two row blocks of gate and of up; NMAT = 1: four
// row blocks) and multiplies each by the three digit planes of all 32 tokens:
// 12 MFMAs per 32-code chunk for 3 LDS operand reads and 28 VALU operations of
// decoding.  The digits of a 128-code group (12 KB) are gathered by
// direct-to-LDS DMA, one chunk per wave, into two stages; the codes go from
// memory to registers, both a group ahead.  192 accumulator registers leave
// two waves per SIMD.
// Blocks of one XCD (blockIdx % 8) take consecutive tiles, row blocks first:
// an expert's weights are read into one L2.
constexpr int kGroupBytes = 4 * 96;              // digits of 128 codes of a token
constexpr int kStage = kGroupTok * kGroupBytes;  // one 128-code group of a tile

template <int NMAT>
__global__ __launch_bounds__(kGemmThreads, 2) void k_moe_gemm(GroupedArgs a) {
  constexpr int RF = 4 / NMAT;  // 32-row blocks per wave
  __shared__ __align__(1024) uint8_t ring[2][kStage];
  const int nt = *a.ntiles, per = (nt + 7) / 8;
  const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
  const int jt = j / a.row_blocks, tile = xcd * per + jt;
  if (jt >= per || tile >= nt) return;
  const int4 ti = a.tiles[tile];
  const int expert = ti.x, ntok = ti.z;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, half = lane >> 5;
  const int m0 = ((j - jt * a.row_blocks) * 4 + wave) * 32 * RF;
  const bool wave_ok = m0 < a.M;
  const int bpr = a.K >> 2, ng = a.K >> 7;

  const int slot = a.slots[ti.y + min(n, ntok - 1)];  // tokens past the tile repeat its last
  const uint32_t src = (uint32_t)(slot / a.src_div) * a.pitch;
  // Digits in LDS: 8 tokens x 128 bytes per DMA instruction (whole lines),
  // token t's 16-byte piece q at piece q ^ (t / 2) of its line, so that the 16
  // tokens of an operand read at one piece fall on different banks.
  const int dma_tok = wave * 8 + (lane >> 3);
  const uint32_t dma_src = (uint32_t)__shfl((int)src, dma_tok) + (((lane & 7) ^ ((dma_tok >> 1) & 7)) << 4);
  const uint32_t b_off = (n >> 3) * (kGroupBytes * 8) + (n & 7) * 128 + ((half ^ ((n >> 1) & 7)) << 4);
  const uint32_t ring_u = lds_u32((const lds_char *)&ring[0][0]);
  auto issue = [&](int g) {
    const uint8_t *base = a.dig + g * kGroupBytes;
    const uint32_t dst = ring_u + (g & 1) * kStage + wave * kGroupBytes * 8;
#pragma unroll
    for (int l = 0; l < 3; ++l) dma16(base + l * 128, dma_src, dst + l * 1024);
  };
  uint32_t aoff[RF];
#pragma unroll
  for (int r = 0; r < RF; ++r) aoff[r] = (uint32_t)(min(m0 + 32 * r + n, a.M - 1) * bpr + 16 * half);
  const uint8_t *wb[NMAT];
#pragma unroll
  for (int i = 0; i < NMAT; ++i) wb[i] = a.w[i] + expert * a.w_stride;
  u32x4_t cur[4], nxt[4];
  auto load = [&](int g, u32x4_t (&d)[4]) {
#pragma unroll
    for (int f = 0; f < 4; ++f)
      d[f] = *reinterpret_cast<const u32x4_t *>(wb[f / RF] + (aoff[f % RF] + (uint32_t)g * 32));
  };

  i32x16_t acc[4][3];
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int p = 0; p < 3; ++p) acc[f][p] = i32x16_t{};
  issue(0);
  load(0, nxt);
  for (int g = 0; g < ng; ++g) {
#pragma unroll
    for (int f = 0; f < 4; ++f) cur[f] = nxt[f];
    // this wave's share of the group has landed and its reads of the other
    // stage have returned; after the barrier, everyone's
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (g + 1 < ng) {
      issue(g + 1);
      load(g + 1, nxt);
    }
    if (!wave_ok) continue;
    const uint8_t *st = ring[g & 1];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      i32x4_t b[3];
#pragma unroll
      for (int p = 0; p < 3; ++p)  // pieces 2 (3 c + p) + half of the group's 24
        b[p] = *reinterpret_cast<const i32x4_t *>(st + ((3 * c + p) >> 2) * 1024 + (b_off ^ (((3 * c + p) & 3) << 5)));
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const i32x4_t codes = decode_codes(cur[f][c]);
#pragma unroll
        for (int p = 0; p < 3; ++p)
          acc[f][p] = __builtin_amdgcn_mfma_i32_32x32x32_i8(codes, b[p], acc[f][p], 0, 0, 0);
      }
    }
  }
  if (!wave_ok || n >= ntok) return;
  // The lane's token and rows: the three digit sums of an output sit in the
  // same register of the three accumulators.
  const DigitMeta meta = *reinterpret_cast<const DigitMeta *>(a.dig + (int64_t)src + 3 * (int64_t)a.K);
  const double qsum = (double)meta.qsum;
  const double unscale = meta.e == kBadExp ? __builtin_nan("") : ldexp(1.0, -meta.e);
  float *out = a.out + (int64_t)slot * a.ld_out;
#pragma unroll
  for (int r = 0; r < RF; ++r)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = m0 + 32 * r + 8 * q + 4 * half;
      if (row >= a.M) continue;  // M % 4 == 0: whole groups of four
      floatx4_t y[NMAT];
#pragma unroll
      for (int i = 0; i < NMAT; ++i) {
        const floatx4_t sc = *reinterpret_cast<const floatx4_t *>(a.scale[i] + expert * a.s_stride + row);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int f = i * RF + r, x = 4 * q + k;
          // exact in f64: |sum| < 2^53, unscale a power of two
          const double tot = __builtin_fma((double)acc[f][2][x], 65536.0,
                                           __builtin_fma((double)acc[f][1][x], 256.0, (double)acc[f][0][x]));
          y[i][k] = (float)((tot - qsum) * unscale) * sc[k];
        }
      }
      if constexpr (NMAT == 2) {
#pragma unroll
        for (int k = 0; k < 4; ++k) y[0][k] = (y[0][k] * (1.0f / (1.0f + expf(-y[0][k])))) * y[1][k];
      }
      *reinterpret_cast<floatx4_t *>(out + row) = y[0];
    }
}

template <int NMAT>
qmla_status launch_gemm(GroupedArgs a, int max_tiles, hipStream_t s) {
  constexpr int block_rows = 4 * 32 * (4 / NMAT);
  a.row_blocks = (a.M + block_rows - 1) / block_rows;
  const int64_t grid = (int64_t)((max_tiles + 7) / 8) * 8 * a.row_blocks;
  k_moe_gemm<NMAT><<<dim3((unsigned)grid), dim3(kGemmThreads), 0, s>>>(a);
  QMLA_LAUNCH_CHECK("k_moe_gemm");
  return QMLA_OK;
}

size_t route_lds_bytes(int E, int H) { return (size_t)kRouteTok * ((size_t)E + H) * sizeof(float); }

}  // namespace

int moe_grouped_max_tiles(int P, int E) { return P / kGroupTok + E; }

bool moe_grouped_supported(const qmla_moe_config &c, int32_t T) {
  const int64_t P = (int64_t)T * c.top_k, H = c.hidden_dim, I = c.intermediate_dim;
  return P >= moe_grouped_min_pairs(c.num_experts) && H <= kGroupedMaxK && I <= kGroupedMaxK &&
         route_lds_bytes(c.num_experts, c.hidden_dim) <= 96 * 1024 &&
         P * std::max(H, I) * 4 < (int64_t)1 << 32 && H * I / 4 < (int64_t)1 << 31;
}

qmla_status launch_moe_grouped_route(const qmla_moe_config &c, const float *xs, int T, const float *gw,
                                     int32_t *sel, float *selw, int32_t *user_idx, float *user_w,
                                     uint8_t *xdig, hipStream_t s) {
  const size_t lds = route_lds_bytes(c.num_experts, c.hidden_dim);
  QMLA_TRY(ensure_dynamic_lds((const void *)k_moe_route_quant, lds));
  k_moe_route_quant<<<dim3((T + kRouteTok - 1) / kRouteTok), dim3(kRouteThreads), lds, s>>>(
      xs, gw, T, c.num_experts, c.hidden_dim, c.top_k, sel, selw, user_idx, user_w, xdig,
      (uint32_t)c.hidden_dim * 4);
  QMLA_LAUNCH_CHECK("k_moe_route_quant");
  return QMLA_OK;
}

qmla_status launch_moe_grouped_experts(const MoeGrouped &m, hipStream_t s) {
  const qmla_moe_config &c = m.cfg;
  const int H = c.hidden_dim, I = c.intermediate_dim;
  const int max_tiles = moe_grouped_max_tiles(m.P, c.num_experts);
  GroupedArgs a{};
  a.w[0] = m.gate_packed;
  a.w[1] = m.up_packed;
  a.scale[0] = m.gate_scales;
  a.scale[1] = m.up_scales;
  a.w_stride = (int64_t)I * (H / 4);
  a.s_stride = I;
  a.M = I;
  a.K = H;
  a.dig = reinterpret_cast<const uint8_t *>(m.y);
  a.pitch = (uint32_t)H * 4;
  a.src_div = c.top_k;
  a.tiles = m.tiles;
  a.ntiles = m.ntiles;
  a.slots = m.slots;
  a.out = m.h;
  a.ld_out = I;
  QMLA_TRY(launch_gemm<2>(a, max_tiles, s));
  if (I <= 16 * kQuantThreads)
    k_moe_quant<1><<<dim3(m.P), dim3(kQuantThreads), 0, s>>>(reinterpret_cast<uint8_t *>(m.h), I);
  else
    k_moe_quant<4><<<dim3(m.P), dim3(kQuantThreads), 0, s>>>(reinterpret_cast<uint8_t *>(m.h), I);
  QMLA_LAUNCH_CHECK("k_moe_quant");
  a.w[0] = a.w[1] = m.down_packed;
  a.scale[0] = a.scale[1] = m.down_scales;
  a.w_stride = (int64_t)H * (I / 4);
  a.s_stride = H;
  a.M = H;
  a.K = I;
  a.dig = reinterpret_cast<const uint8_t *>(m.h);
  a.pitch = (uint32_t)I * 4;
  a.src_div = 1;
  a.out = m.y;
  a.ld_out = H;
  return launch_gemm<1>(a, max_tiles, s);
}

}  // namespace qmla
