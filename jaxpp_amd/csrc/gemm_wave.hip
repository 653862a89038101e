// bf16 products of few tiles: C[m,n] = epilogue(sum_k A[m,k] Bop[n,k]), A's contraction index
// contiguous (forward and input-gradient products).
//
// A workgroup owns BM x 64 outputs, 32 or 64 rows; its W waves each multiply the whole tile over every
// W-th K-step of 64 and their sums meet in LDS, in wave order.  With fewer tiles than CUs a product's
// time is one tile's, and a tile whose waves share their operands in LDS is a chain of
// latencies: barrier, fragment reads, copies, K-step after K-step.  Here every wave copies its own
// steps into LDS of its own and waits for nothing but them: no barrier before the sums, and the
// copies of the waves keep the CU's path to memory (64 bytes a cycle) busy, which is then what
// bounds a tile of 32 rows: 12 KB a K-step, 192 cycles.  512 x 1024 x 4096 (256 tiles) 17.4 -> 13.9 us, 512 x
// 1024 x 1024 9.0 -> 7.4, 256 x 256 x 768 7.2 -> 5.7, 128 x 128 x 128 5.0 -> 4.3, against 64 x 64 tiles
// shared by two wave groups; without the copies past the end (3 of 7 at K = 1024) the first 10.3 where that
// product runs by itself.  (Operands from L2 straight into fragments, without LDS: 28 us, a load of 16
// rows x 64 bytes holds the path far longer than its kilobyte.)
// Tiles of 64 rows, 16 KB a K-step, for up to twice the outputs: four waves with two stages each, which
// is all that fits, and the copies between the MFMAs; 512 x 2048 outputs at K = 11264 / 5632 / 2048 46 -> 39 / 27
// -> 25.7 / 9.6 -> 9.0 us against the tiles shared by two wave groups, 0.85 - 0.95 over 70 random shapes.
// With a GELU or its derivative eight waves with one stage each, whose epilogue has twice the
// threads: 0.85 - 0.95 (GELU) and 0.93 - 1.0 from 9 K-steps on, 1.0 - 1.1 below.  (Three stages of three waves 41.6 us
// for the first, two of five 41.4, eight waves 37.8 but 12.1 instead of 11.8 at K = 3072.)
//
// The operands' LDS images and the fragments read from them are those of gemm.hip (DmaTile), the
// n side on the MFMA's A port: lane (c = lane % 16, g = lane / 16) ends up with row 16 i + c and
// columns 16 j + 4 g + r of tile (i, j).
#include <math.h>

#include "gemm_wave.h"

namespace {

constexpr int PITCH = 68;                      // floats of a row of the sums

// BM: rows of a tile; W: waves, one or two per SIMD; NS: stages of a wave
template <bool TB, int EPI, int BM, int W, int NS>
__global__ __launch_bounds__(64 * W) void gemm_wave_kernel(GemmWave p) {
  constexpr int TM = BM / 16;
  using TileA = DmaTile<BM, false, 1>;
  using TileB = DmaTile<64, TB, 1>;
  constexpr int STAGE = TileA::BYTES + TileB::BYTES, COPIES = TileA::INSTS + TileB::INSTS;
  extern __shared__ __align__(1024) uint8_t smem[];   // [W][NS][STAGE]; then [W][BM][PITCH] floats
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Consecutive workgroups go to the eight XCDs in turn, each with an L2 of its own: every XCD
  // takes a run of tiles, 256 rows at a time, so that it reads a part of both operands.
  const int tiles_n = p.n / 64, tiles_m = p.m / BM;
  // (64 rows: the first XCDs one tile more where the number is not a multiple of 8 - 252 tiles as they come
  // took 1.16 of the time of the tiles shared by wave groups, in runs 0.92.  The few scalar
  // instructions more cost products of 32 rows 0.2 us each, a row of 512 tokens 1 %.)
  int pid = blockIdx.x;
  if constexpr (BM == 64) {
    const int nwg = gridDim.x, x = pid & 7;
    pid = x * (nwg >> 3) + min(x, nwg & 7) + (pid >> 3);
  } else if ((gridDim.x & 7) == 0) {
    pid = (pid & 7) * (gridDim.x >> 3) + (pid >> 3);
  }
  const int rows = 256 / BM, first = pid / (rows * tiles_n) * rows, rows_here = min(tiles_m - first, rows);
  const int within = pid - first * tiles_n;
  const long m0 = (long)(first + within % rows_here) * BM, n0 = (long)(within / rows_here) * 64;

  // the epilogue's share of this thread: 8 columns of a row, and of every STEP-th row behind it; what
  // they are added to or multiplied with arrives during the contraction
  constexpr int STEP = 8 * W, MINE = (BM + STEP - 1) / STEP;
  const int row = tid >> 3;
  const long ocol = n0 + (tid & 7) * 8;
  const bf16_t* const pre_src = EPI == JPP_EPI_DGELU ? p.aux : EPI == JPP_EPI_BF16 ? p.resid : nullptr;
  const long pre_ld = EPI == JPP_EPI_DGELU ? p.ldaux : p.ldresid;
  uint4 pre[MINE], bias = make_uint4(0, 0, 0, 0);
#pragma unroll
  for (int q = 0; q < MINE; ++q) {
    pre[q] = make_uint4(0, 0, 0, 0);
    if (pre_src && (BM % STEP == 0 || row + q * STEP < BM)) pre[q] = *(const uint4*)(pre_src + (m0 + row + q * STEP) * pre_ld + ocol);
  }
  if (p.bias) bias = *(const uint4*)(p.bias + ocol);

  f32x4 acc[TM][4];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = (p.k / 64 - wave + W - 1) / W;   // wave, wave + W, ...
  if (steps > 0) {
    typename TileA::Offsets offa;
    typename TileB::Offsets offb;
    TileA::offsets(offa, p.lda, 0, lane);
    TileB::offsets(offb, p.ldb, 0, lane);
    const long step_b = TB ? 64 * p.ldb : 64;
    const bf16_t* const pa = p.a + m0 * p.lda + wave * 64;
    const bf16_t* const pb = p.b + (TB ? n0 : n0 * p.ldb) + wave * step_b;
    const uint8_t* const stages = smem + wave * (NS * STAGE);
    const uint32_t lds0 = lds_address(stages);
    auto copy = [&](int stage, int t) {
      if (t >= steps) return;
      const long at = t;
      TileA::template issue<0, TileA::INSTS>(uniform_ptr(pa + at * (W * 64)), offa, lds0 + stage * STAGE, 0);
      TileB::template issue<0, TileB::INSTS>(uniform_ptr(pb + at * W * step_b), offb,
                                             lds0 + stage * STAGE + TileA::BYTES, 0);
    };
#pragma unroll
    for (int s = 0; s < NS; ++s) copy(s, s);
    int st = 0;
    for (int t = 0; t < steps; ++t) {
      dma_wait_groups<COPIES, NS - 1>(steps - 1 - t);   // (copies land in order: this step's have)
      const uint8_t* const sa = stages + st * STAGE;
      const uint8_t* const sb = sa + TileA::BYTES;
      bf16x8 fa[2][TM], fb[2][4];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
#pragma unroll
        for (int j = 0; j < 4; ++j) fb[k][j] = TileB::frag16(sb, 16 * j, k, lane);
#pragma unroll
        for (int i = 0; i < TM; ++i) fa[k][i] = TileA::frag16(sa, 16 * i, k, lane);
      }
      // every fragment is in registers: the stage can be filled again - of 32 rows at once, of 64
      // between the MFMAs, which the copies would keep waiting for the path (a wave issues in
      // order; with 32 rows that order costs a row of products of 512 tokens 1.5 %)
      lds_wait_all();
      constexpr int PARTS = BM == 32 ? 1 : 2 * TM, PER = COPIES / PARTS;
      static_assert(COPIES % PARTS == 0, "copies split evenly over the rows of MFMAs");
      auto refill = [&](int part) {
        if (t + NS >= steps) return;
        const bf16_t* const na = uniform_ptr(pa + (long)(t + NS) * (W * 64));
        const bf16_t* const nb = uniform_ptr(pb + (long)(t + NS) * W * step_b);
#pragma unroll
        for (int q = part * PER; q < part * PER + PER; ++q) {
          if (q < TileA::INSTS) dma_load16(na, offa[min(q, TileA::INSTS - 1)], lds0 + st * STAGE + q * 1024);
          else dma_load16(nb, offb[max(q - TileA::INSTS, 0)], lds0 + st * STAGE + q * 1024);
        }
      };
      if (PARTS == 1) refill(0);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        if constexpr (PARTS == 1) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[k][j], fa[k][i], acc[i][j], 0, 0, 0);
        } else {
#pragma unroll
          for (int i = 0; i < TM; ++i) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[k][j], fa[k][i], acc[i][j], 0, 0, 0);
            refill(k * TM + i);
          }
        }
      }
      st = st + 1 == NS ? 0 : st + 1;
    }
  }
  __syncthreads();
  float* const part = (float*)smem;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *(f32x4*)(part + (wave * BM + 16 * i + c) * PITCH + 16 * j + 4 * g) = acc[i][j];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < MINE; ++q) {
    const int r = row + q * STEP;
    if (BM % STEP && r >= BM) break;
    const float* src = part + r * PITCH + (tid & 7) * 8;
    f32x4 lo = *(const f32x4*)src, hi = *(const f32x4*)(src + 4);
#pragma unroll
    for (int w = 1; w < W; ++w) {
      lo += *(const f32x4*)(src + w * BM * PITCH);
      hi += *(const f32x4*)(src + w * BM * PITCH + 4);
    }
    float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}, u[8];
    if (p.bias) {
      unpack8(bias, u);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += u[e];
    }
    unpack8(pre[q], u);
    if constexpr (EPI == JPP_EPI_BF16) {
      if (p.resid) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += u[e];
      }
    } else if constexpr (EPI == JPP_EPI_DGELU) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] *= gelu_grad_f(u[e], p.gelu_tanh);
    } else {
      float gl[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) gl[e] = gelu_f(v[e], p.gelu_tanh);
      *(uint4*)(p.c2 + (m0 + r) * p.ldc2 + ocol) = pack8(gl);
    }
    *(uint4*)(p.c + (m0 + r) * p.ldc + ocol) = pack8(v);
  }
}

template <bool TB, int EPI, int BM, int W, int NS>
int launch(hipStream_t st, const GemmWave& p) {
  constexpr int LOOP = W * NS * (BM + 64) * 128, SUMS = W * BM * PITCH * 4, SMEM = LOOP > SUMS ? LOOP : SUMS;
  static_assert(SMEM <= 160 * 1024, "LDS of one CU");
  auto kern = gemm_wave_kernel<TB, EPI, BM, W, NS>;
  static std::once_flag configured;   // (the limit is sticky per kernel)
  static hipError_t configure_rc = hipSuccess;
  std::call_once(configured, [&] {
    configure_rc = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
  });
  JPP_CHECK_HIP(configure_rc);
  hipLaunchKernelGGL(kern, dim3((unsigned)((p.m / BM) * (p.n / 64))), dim3(64 * W), SMEM, st, p);
  JPP_LAUNCH_CHECK();
  return JPP_OK;
}

template <bool TB, int EPI>
int launch_rows(hipStream_t st, const GemmWave& p, int rows) {
  if (rows == 32) return launch<TB, EPI, 32, 4, 3>(st, p);
  return EPI == JPP_EPI_BF16 ? launch<TB, EPI, 64, 4, 2>(st, p) : launch<TB, EPI, 64, 8, 1>(st, p);
}

}  // namespace

int launch_gemm_wave(hipStream_t st, const GemmWave& p, bool tb, int epi, int rows) {
  const bool plain = epi == JPP_EPI_BF16;
  if (tb) return plain ? launch_rows<true, JPP_EPI_BF16>(st, p, rows) : launch_rows<true, JPP_EPI_GELU>(st, p, rows);
  return plain ? launch_rows<false, JPP_EPI_BF16>(st, p, rows) : launch_rows<false, JPP_EPI_DGELU>(st, p, rows);
}
