// rows_gemm.hip -- the projections of an MLA layer call over 1 .. 127 token
// rows (MlaAttention::forward_prefill, src/model.rs:197-249, on a short
// prompt): y[m][n] = sum_k x[m][k] W[n][k] in f32 on v_mfma_f32_32x32x2_f32,
// products and sums exact to f32 rounding, with the layout work of
// split_gemm.hip's epilogues.
//
// Bound: the f32 MFMA rate, from about 64 rows; below, the stream of the
// weights.  All M rows of a product go to one block, so each weight is read
// once; a block owns 64 outputs and one of ksplit slices of K, and its four
// waves split that slice again, so that the 57 tiles of the 3648-wide
// q_proj | kv_a fill 228 CUs at ksplit = 4.  A wave streams 16 k of its 64
// weight rows and M token rows at a time through three LDS stages of its own
// by direct-to-LDS DMA, two groups in flight, with no barrier in the loop.
// (Straight to registers, a load touches 32 rows of 16 bytes, 64 clocks of
// address work: q_proj | kv_a at 77 rows takes 25.3 us that way, 20.8 with
// the DMA, which covers 16 rows of 64 bytes; its MFMAs alone take 10.2.)  The four waves' tiles are added
// through LDS, the slices' partial sums by k_sg_reduce, which also applies
// bias and epilogue.
#include <type_traits>

#include "mfma_pipe.hpp"

namespace qmla {

namespace {

using namespace pipe;

constexpr int kRgWaves = 4, kRgStages = 3;
constexpr int kRgK = 16;   // k per stage
constexpr int kRgLd = 36;  // floats per staged row of a 32 x 32 tile (padded)

// Bytes of a stage: 64 weight rows and 32 MB token rows (f32, or bf16).
constexpr int rg_stage(int MB, bool XB16) { return 64 * 64 + 32 * MB * (XB16 ? 32 : 64); }

// In a stage a row's 16-byte pieces (4, or 2 of bf16) are permuted by its
// index, which spreads the 16 rows that a read covers over all banks.
// XB16: x is the bf16 attention context (x_heads), widened as it is read.
template <int MB, bool XB16>
__global__ __launch_bounds__(kRgWaves * 64) void k_rows_gemm(RowsGemmArgs a) {
  constexpr int STAGE = rg_stage(MB, XB16);
  constexpr int XD = XB16 ? MB : 2 * MB;  // DMA instructions per stage: 4 + XD
  extern __shared__ __attribute__((aligned(1024))) uint8_t ring[];
  const SplitGemmArgs &g = a.g;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = lane & 31, h = lane >> 5;
  const int n0 = blockIdx.x * 64;
  // this wave's groups of 16 k: [c0, c0 + NC), even shares
  const int KC = g.K / kRgK, sl = blockIdx.y * kRgWaves + wave, S = g.ksplit * kRgWaves;
  const int c0 = (int)((int64_t)KC * sl / S), NC = (int)((int64_t)KC * (sl + 1) / S) - c0;

  // per-lane DMA offsets; rows past N or M re-read the last one (their
  // outputs are dropped)
  uint32_t wo[4], xo[XD];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 16 * i + (lane >> 2);
    wo[i] = (uint32_t)(min(r, g.N - 1 - n0) * g.K * 4 + (((lane & 3) ^ ((r >> 2) & 3)) << 4));
  }
#pragma unroll
  for (int i = 0; i < XD; ++i) {
    const int r = XB16 ? 32 * i + (lane >> 1) : 16 * i + (lane >> 2);
    const int m = min(r, g.M - 1);
    int64_t e;
    if (g.x_heads) {
      const int b = m / g.seq;
      e = ((int64_t)b * g.heads * g.seq + (m - b * g.seq)) * g.dv;
    } else {
      e = (int64_t)m * g.ldx;
    }
    xo[i] = XB16 ? (uint32_t)(e * 2 + (((lane & 1) ^ ((r >> 3) & 1)) << 4))
                 : (uint32_t)(e * 4 + (((lane & 3) ^ ((r >> 2) & 3)) << 4));
  }
  const uint8_t *wb = reinterpret_cast<const uint8_t *>(a.w + (int64_t)n0 * g.K);
  const uint8_t *xb = reinterpret_cast<const uint8_t *>(g.x);
  uint8_t *my = ring + wave * (kRgStages * STAGE);
  const uint32_t my_u = lds_u32((const lds_char *)my);
  auto issue = [&](int c) __attribute__((always_inline)) {
    const int k = (c0 + c) * kRgK;
    const uint32_t st = my_u + (uint32_t)(c % kRgStages * STAGE);
#pragma unroll
    for (int i = 0; i < 4; ++i) dma16(wb + (int64_t)k * 4, wo[i], st + i * 1024);
    int64_t ke = k;
    if (g.x_heads) {  // dv % 16 == 0: a group lies in one head
      const int hd = k / g.dv;
      ke = (int64_t)hd * g.seq * g.dv + (k - hd * g.dv);
    }
#pragma unroll
    for (int i = 0; i < XD; ++i) dma16(xb + ke * (XB16 ? 2 : 4), xo[i], st + 4096 + i * 1024);
  };

  floatx16_t acc[2][MB];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  if (NC > 0) issue(0);
  if (NC > 1) issue(1);
  for (int c = 0; c < NC; ++c) {
    // group c has landed, and the reads of group c - 1, whose stage group
    // c + 2 takes, have returned
    if (c + 1 < NC)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(4 + XD) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    // the group's operands, then the next DMA under their latency
    const uint8_t *st = my + c % kRgStages * STAGE;
    floatx4_t w[2][2], x[2][MB];
    u32x2_t x2[2][MB];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int po = ((2 * q + h) ^ ((row >> 2) & 3)) << 4;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        w[q][i] = *reinterpret_cast<const floatx4_t *>(st + (32 * i + row) * 64 + po);
#pragma unroll
      for (int j = 0; j < MB; ++j)
        if constexpr (XB16)
          x2[q][j] = *reinterpret_cast<const u32x2_t *>(
              st + 4096 + (32 * j + row) * 32 + ((q ^ ((row >> 3) & 1)) << 4) + 8 * h);
        else
          x[q][j] = *reinterpret_cast<const floatx4_t *>(st + 4096 + (32 * j + row) * 64 + po);
    }
    if (c + 2 < NC) issue(c + 2);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if constexpr (XB16)
#pragma unroll
        for (int j = 0; j < MB; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            x[q][j][e] = __builtin_bit_cast(
                float, e & 1 ? x2[q][j][e >> 1] & 0xffff0000u : x2[q][j][e >> 1] << 16);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < MB; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(w[q][i][e], x[q][j][e], acc[i][j], 0,
                                                             0, 0);
    }
  }

  // element e of lane l: output 8 (e / 4) + 4 (l / 32) + e % 4, row l % 32
  float *part = g.part + (int64_t)blockIdx.y * g.M * g.N;
  float *red = reinterpret_cast<float *>(ring);  // two tiles of each wave in turn
  constexpr int TILE = 32 * kRgLd;
  static_assert(2 * kRgWaves * TILE * 4 <= kRgWaves * kRgStages * STAGE, "ring holds the tiles");
  const int rm = threadIdx.x >> 3, rn = 4 * (threadIdx.x & 7);
  __syncthreads();  // every wave is done with its ring
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j) {
      float *rd = red + ((i * MB + j) & 1) * (kRgWaves * TILE);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<floatx4_t *>(rd + wave * TILE + row * kRgLd + 8 * q + 4 * h) =
            floatx4_t{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                      acc[i][j][4 * q + 3]};
      __syncthreads();
      floatx4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < kRgWaves; ++w)
        v += *reinterpret_cast<const floatx4_t *>(rd + w * TILE + rm * kRgLd + rn);
      const int m = 32 * j + rm, n = n0 + 32 * i + rn;  // N % 4 == 0
      if (m < g.M && n < g.N) *reinterpret_cast<floatx4_t *>(part + (int64_t)m * g.N + n) = v;
    }
}

template <int MB, bool XB16>
qmla_status go(const RowsGemmArgs &a, hipStream_t s) {
  const size_t lds = (size_t)kRgWaves * kRgStages * rg_stage(MB, XB16);
  QMLA_TRY(ensure_dynamic_lds((const void *)k_rows_gemm<MB, XB16>, lds));
  k_rows_gemm<MB, XB16><<<dim3((unsigned)((a.g.N + 63) / 64), (unsigned)a.g.ksplit),
                          dim3(kRgWaves * 64), lds, s>>>(a);
  QMLA_LAUNCH_CHECK("k_rows_gemm");
  return launch_sg_reduce(a.g, s);
}

// K slices: powers of two up to 8 while the blocks stay within one round of
// the device (twice as many: 1 x 77 tokens 74.3 -> 78.3 us, half 74 -> 101)
// and a wave keeps at least two groups of k.
int rows_gemm_slices(int N, int K) {
  const int tiles = (N + 63) / 64;
  int s = 1;
  while (s < 8 && tiles * s * 2 <= 256 && K / (2 * s * kRgWaves) >= 2 * kRgK) s *= 2;
  return s;
}

}  // namespace

size_t rows_gemm_part_bytes(int M, int N, int K) {
  return (size_t)rows_gemm_slices(N, K) * M * N * sizeof(float);
}

qmla_status launch_rows_gemm(const RowsGemmArgs &a0, hipStream_t s) {
  RowsGemmArgs a = a0;
  const auto &g = a.g;
  QMLA_REQUIRE(g.M >= 1 && g.M <= 128 && split_gemm_supported(g.N, g.K) && g.part && g.seq > 0 &&
                   g.K <= 1 << 22 && g.ldx <= 1 << 22,
               QMLA_ERR_UNSUPPORTED, "rows GEMM M %d N %d K %d", g.M, g.N, g.K);
  QMLA_REQUIRE(!g.x_heads || (g.dv % kRgK == 0 && g.K == g.heads * g.dv), QMLA_ERR_SHAPE,
               "rows GEMM head-major x: dv %d, K %d", g.dv, g.K);
  QMLA_REQUIRE(g.x_heads || !g.x_bf16, QMLA_ERR_SHAPE, "rows GEMM: bf16 rows");
  a.g.ksplit = rows_gemm_slices(g.N, g.K);
  auto pick = [&](auto b16) -> qmla_status {
    constexpr bool XB16 = decltype(b16)::value;
    switch ((g.M + 31) / 32) {
      case 1: return go<1, XB16>(a, s);
      case 2: return go<2, XB16>(a, s);
      case 3: return go<3, XB16>(a, s);
      default: return go<4, XB16>(a, s);
    }
  };
  return g.x_bf16 ? pick(std::true_type{}) : pick(std::false_type{});
}

}  // namespace qmla
