// The layer's operators on fp32 tensors: the full-precision flavour of a stage, as the
// reference's own CPU-runnable configuration uses it (BERT-style stack of hidden 256 in
// float32, tests/test_transformations.py:42-93 builds its model in float32 too).  Same
// argument structs as the bf16 entry points with every bf16 tensor replaced by an f32 one.
//
// These kernels serve small problems whose results must hold 1e-4 against an fp32 CPU run:
// fp32 arithmetic throughout, the contractions on the fp32 matrix instruction, every sum in an
// order that the shapes fix.
#include <limits.h>
#include <math.h>
#include <string.h>

#include <mutex>

#include "common.h"

namespace {

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

__device__ __forceinline__ float gelu32(float u, int tanh_form) {
  if (tanh_form) {
    const float t = tanhf(0.7978845608028654f * (u + 0.044715f * u * u * u));
    return 0.5f * u * (1.0f + t);
  }
  return 0.5f * u * (1.0f + erff(u * 0.7071067811865476f));
}

__device__ __forceinline__ float gelu_grad32(float u, int tanh_form) {
  if (tanh_form) {
    const float t = tanhf(0.7978845608028654f * (u + 0.044715f * u * u * u));
    return 0.5f * (1.0f + t) +
           0.5f * u * (1.0f - t * t) * 0.7978845608028654f * (1.0f + 0.134145f * u * u);
  }
  return 0.5f * (1.0f + erff(u * 0.7071067811865476f)) +
         u * expf(-0.5f * u * u) * 0.3989422804014327f;
}

__device__ __forceinline__ float swiglu32(float g, float u) { return g / (1.0f + expf(-g)) * u; }
__device__ __forceinline__ void swiglu_grad32(float g, float u, float d, float& dg, float& du) {
  const float sg = 1.0f / (1.0f + expf(-g));
  dg = d * u * sg * (1.0f + g * (1.0f - sg));
  du = d * g * sg;
}

// ---------------------------------------------------------------------------
// C[m,n] = epilogue(sum_k Aop[m,k] Bop[n,k]); operand orientations as jpp_gemm_bf16
// ---------------------------------------------------------------------------
struct SgemmParams {
  const float* a;
  const float* b;
  float* c;
  float* c2;
  const float* bias;
  const float* resid;
  const float* aux;
  int m, n, k;
  long lda, ldb, ldc, ldc2, ldresid, ldaux;
  int ta, tb, epi, gelu_tanh;
  // grouped problems, as for the bf16 GEMM: seg[0..n_seg] are row offsets (multiples of 64)
  const int* seg;
  int n_seg, group_mode;
  long stride_b, stride_c;
};

// operand vectors: 16 (8) bytes from addresses of which 4-byte alignment is known
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2_u __attribute__((ext_vector_type(2), aligned(4)));

// One wave's fragments of an operand for 16 contraction elements: T subtiles of 16 rows, for
// v_mfma_f32_16x16x4_f32.  Lane l (c = l % 16, g = l / 16) supplies row c of subtile i with
// contraction element 4 g + s to MFMA s; any order serves as long as both operands share it,
// and this one makes every load a vector of the operand's contiguous index:
//   SLOW = false  [rows][k]: row 16 i + c, elements 4 g .. 4 g + 3 in one load per subtile
//   SLOW = true   [k][rows]: rows T c .. T c + T - 1 (row T c + i belongs to subtile i) of
//                 contraction element 4 g + s in one load per s
template <int T, bool SLOW>
struct Frag32 {
  float v[T][4];
  __device__ __forceinline__ void load(const float* p, long ld) {
    if constexpr (!SLOW) {
#pragma unroll
      for (int i = 0; i < T; ++i) {
        const f32x4_u q = *(const f32x4_u*)(p + 16 * i * ld);
#pragma unroll
        for (int s = 0; s < 4; ++s) v[i][s] = q[s];
      }
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if constexpr (T == 4) {
          const f32x4_u q = *(const f32x4_u*)(p + s * ld);
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i][s] = q[i];
        } else if constexpr (T == 2) {
          const f32x2_u q = *(const f32x2_u*)(p + s * ld);
          v[0][s] = q[0];
          v[1][s] = q[1];
        } else {
          v[0][s] = p[s * ld];
        }
      }
    }
  }
  // this lane's first element of the tile whose first row and contraction element are `p`
  static __device__ __forceinline__ const float* lane_ptr(const float* p, long ld, int c, int g) {
    return SLOW ? p + 4 * g * ld + T * c : p + c * ld + 4 * g;
  }
};

template <int BM>
constexpr int kStages32 = BM == 16 ? 3 : 2;   // (what fits beside the sums)

// A workgroup owns BM x 64 outputs; its four waves each multiply the whole tile over every
// fourth step of 16 contraction elements, and their four sums meet in LDS in wave order.
// These products are small (512 x 256 x 256 and a few times that): what bounds them is latency,
// so the work is spread over as many CUs as the tile allows and inside a CU over the
// contraction, and operands go from L2 straight into MFMA fragments - no barrier and no LDS
// before the sums, D steps of loads in flight per wave.  v_mfma_f32_16x16x4_f32 accumulates as
// a chain of fused multiply-adds does, at twice the rate of v_fma_f32; the four shorter chains
// halve the distance to a float64 sum (5.7e-7 -> 2.9e-7 at k = 1024).  512 x 256 outputs, k = 256
// and 1024, take 7.3 us on average; the 64 x 64 tile of 16 x 16 threads in its place, one barrier
// pair per 16 contraction elements on 32 CUs, and attention with a pair of lanes per row made a
// two-layer row of eight microbatches of 512 tokens 30.0 ms, now 1.70 ms.
//
// STAGED (both contraction indices contiguous): every wave copies its own steps, 32 elements of
// the contraction at a time, into LDS of its own and reads the fragments there, with no barrier
// either.  A fragment loaded from memory directly touches 16 rows with 64 bytes each, and the
// CU's path takes such a load far longer than one of eight whole lines; of the operands of the
// other orientations one is read along its rows anyway (512 x 256, k = 256 to 1024: 10.3 -> 7.0 us
// on average).  (A 32-element step is 128 bytes a row:
// the LDS image is that of a bf16 tile of 64.)
template <int BM, bool TA, bool TB, bool STAGED>
__device__ __forceinline__ void sgemm_tile(SgemmParams p, int blk) {
  constexpr int TM = BM / 16, TN = 4, D = BM == 64 ? 2 : 4, PITCH = 68;
  static_assert(!STAGED || (!TA && !TB && BM <= 32), "staged: both operands [rows][k], two tiles' LDS");
  extern __shared__ __align__(1024) uint8_t smem[];   // (STAGED) [4 waves][stages][BM + 64 rows of 128 bytes]
  __shared__ float part[2][4][16 * PITCH];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_n = p.n / 64;
  const long m0 = (long)(blk / tiles_n) * BM, n0 = (long)(blk % tiles_n) * 64;
  if (p.group_mode == JPP_GROUP_M) {
    // rows of A and C are grouped by expert; each group multiplies its own B
    if (m0 >= p.seg[p.n_seg]) return;
    int e = 0;
    while (p.seg[e + 1] <= m0) ++e;
    p.b += (long)e * p.stride_b;
  } else if (p.group_mode == JPP_GROUP_K) {
    // one output per expert (blockIdx.z); the contraction runs over the expert's rows
    const int e = blockIdx.z;
    const long r0 = p.seg[e];
    p.k = p.seg[e + 1] - p.seg[e];
    p.a += r0 * p.lda;
    p.b += r0 * p.ldb;
    p.c += (long)e * p.stride_c;
  }
  // the epilogue's 16 rows at a time: pass i holds subtile i, a thread four columns of a row
  const int er = tid >> 4, eq = (tid & 15) * 4;
  const long col = n0 + eq;
  auto out_row = [&](int i) { return m0 + (TA ? TM * er + i : 16 * i + er); };
  // what the epilogue adds or multiplies with arrives during the contraction
  const float* pre_src = p.epi == JPP_EPI_ACC_F32 ? p.c : p.epi == JPP_EPI_DGELU ? p.aux
                         : p.epi == JPP_EPI_BF16 ? p.resid : nullptr;
  const long pre_ld = p.epi == JPP_EPI_ACC_F32 ? p.ldc : p.epi == JPP_EPI_DGELU ? p.ldaux : p.ldresid;
  f32x4 pre[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
    pre[i] = pre_src ? (f32x4)*(const f32x4_u*)(pre_src + out_row(i) * pre_ld + col) : f32x4{0.f, 0.f, 0.f, 0.f};

  typedef Frag32<TM, TA> FA;
  typedef Frag32<TN, TB> FB;
  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (STAGED) {
    constexpr int NS = kStages32<BM>, STAGE = (BM + 64) * 128;
    using TileA = DmaTile<BM, false, 1>;
    using TileB = DmaTile<64, false, 1>;
    const int steps = (p.k / 32 - wave + 3) / 4;   // wave, wave + 4, ...
    if (steps > 0) {
      typename TileA::Offsets offa;
      typename TileB::Offsets offb;
      TileA::offsets(offa, 2 * p.lda, 0, lane);    // (in 2-byte elements)
      TileB::offsets(offb, 2 * p.ldb, 0, lane);
      const bf16_t* const pa = (const bf16_t*)(p.a + m0 * p.lda + wave * 32);
      const bf16_t* const pb = (const bf16_t*)(p.b + n0 * p.ldb + wave * 32);
      const uint8_t* const stages = smem + wave * (NS * STAGE);
      const uint32_t lds0 = lds_address(stages);
      auto copy = [&](int stage, int t) {
        if (t >= steps) return;
        const long at = t * 256L;
        TileA::template issue<0, TileA::INSTS>(uniform_ptr(pa + at), offa, lds0 + stage * STAGE, 0);
        TileB::template issue<0, TileB::INSTS>(uniform_ptr(pb + at), offb, lds0 + stage * STAGE + BM * 128, 0);
      };
#pragma unroll
      for (int q = 0; q < NS; ++q) copy(q, q);
      int st = 0;
      for (int t = 0; t < steps; ++t) {
        dma_wait_groups<TileA::INSTS + TileB::INSTS, NS - 1>(steps - 1 - t);
        const uint8_t* const sa = stages + st * STAGE;
        f32x4 fa[2][TM], fb[2][TN];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
          for (int j = 0; j < TN; ++j) fb[h][j] = *(const f32x4*)(sa + BM * 128 + slab_off(16 * j + c, 4 * h + g));
#pragma unroll
          for (int i = 0; i < TM; ++i) fa[h][i] = *(const f32x4*)(sa + slab_off(16 * i + c, 4 * h + g));
        }
        lds_wait_all();   // every fragment is in registers: the stage can be filled again
        copy(st, t + NS);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
              for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[h][j][s], fa[h][i][s], acc[i][j], 0, 0, 0);
        st = st + 1 == NS ? 0 : st + 1;
      }
    }
    dma_wait_all();
  }
  const int steps = STAGED ? 0 : (p.k / 16 - wave + 3) / 4;   // wave, wave + 4, ...
  if (steps > 0) {
    const long step_a = TA ? 64 * p.lda : 64, step_b = TB ? 64 * p.ldb : 64;
    const float* pa = FA::lane_ptr(p.a + (TA ? m0 : m0 * p.lda), p.lda, c, g) + wave * (step_a / 4);
    const float* pb = FB::lane_ptr(p.b + (TB ? n0 : n0 * p.ldb), p.ldb, c, g) + wave * (step_b / 4);
    FA fa[D];
    FB fb[D];
#pragma unroll
    for (int u = 0; u < D - 1; ++u) {
      fa[u].load(pa + min(u, steps - 1) * step_a, p.lda);
      fb[u].load(pb + min(u, steps - 1) * step_b, p.ldb);
    }
    for (int t = 0; t < steps; t += D) {
#pragma unroll
      for (int u = 0; u < D; ++u) {
        // (past the end the last step is fetched again, unused)
        const long nt = min(t + u + D - 1, steps - 1);
        fa[(u + D - 1) % D].load(pa + nt * step_a, p.lda);
        fb[(u + D - 1) % D].load(pb + nt * step_b, p.ldb);
        if (t + u < steps) {
#pragma unroll
          for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
              for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[u].v[j][s], fa[u].v[i][s], acc[i][j], 0, 0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    // lane (c, g): row c of subtile i and, of column subtile j, the four indices 4 g + r
    float* mine = &part[i & 1][wave][c * PITCH];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *(f32x4*)(mine + 16 * (TB ? g : j) + 4 * (TB ? j : g)) =
          TB ? f32x4{acc[i][0][j], acc[i][1][j], acc[i][2][j], acc[i][3][j]} : acc[i][j];
    __syncthreads();
    const float* src = &part[i & 1][0][er * PITCH + eq];
    f32x4 v = *(const f32x4*)src;
#pragma unroll
    for (int w = 1; w < 4; ++w) v += *(const f32x4*)(src + w * 16 * PITCH);
    const long row = out_row(i);
    float* const dst = p.c + row * p.ldc + col;
    if (p.epi == JPP_EPI_ACC_F32) {
      *(f32x4_u*)dst = pre[i] + v;
      continue;
    }
    if (p.epi == JPP_EPI_SWIGLU) {
      // a 64-column tile is one block of the interleaved layout: gate features in its first
      // 32 columns (threads eq < 32), the matching up features 32 columns on (lane + 8)
      *(f32x4_u*)dst = v;
      f32x4 s;
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = swiglu32(v[e], __shfl_xor(v[e], 8));
      if (eq < 32) *(f32x4_u*)(p.c2 + row * p.ldc2 + n0 / 2 + eq) = s;
      continue;
    }
    if (p.epi == JPP_EPI_DSWIGLU) {
      // v = d s of features col .. col + 3; gate / up of feature f sit at 64 (f / 32) + f % 32
      // and 32 behind it
      const long at = 64 * (col >> 5) + (col & 31);
      const f32x4 gate = *(const f32x4_u*)(p.aux + row * p.ldaux + at);
      const f32x4 up = *(const f32x4_u*)(p.aux + row * p.ldaux + at + 32);
      f32x4 dg, du;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float x, y;
        swiglu_grad32(gate[e], up[e], v[e], x, y);
        dg[e] = x;
        du[e] = y;
      }
      *(f32x4_u*)(p.c + row * p.ldc + at) = dg;
      *(f32x4_u*)(p.c + row * p.ldc + at + 32) = du;
      continue;
    }
    if (p.bias) v += (f32x4)*(const f32x4_u*)(p.bias + col);
    if (p.epi == JPP_EPI_GELU) {
      f32x4 s;
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = gelu32(v[e], p.gelu_tanh);
      *(f32x4_u*)(p.c2 + row * p.ldc2 + col) = s;
    } else if (p.epi == JPP_EPI_DGELU) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= gelu_grad32(pre[i][e], p.gelu_tanh);
    } else if (p.resid) {
      v += p.epi == JPP_EPI_BF16 ? pre[i] : (f32x4)*(const f32x4_u*)(p.resid + row * p.ldresid + col);
    }
    *(f32x4_u*)dst = v;
  }
}

template <int BM, bool TA, bool TB, bool STAGED>
__global__ __launch_bounds__(256) void sgemm_kernel(SgemmParams p) {
  sgemm_tile<BM, TA, TB, STAGED>(p, blockIdx.x);
}

// Rows of a product's tiles: the tallest that still give every CU one (a taller tile reads its B fewer times).
int tile_rows32(long strips) { return strips >= 4 * 256 ? 64 : strips >= 2 * 256 ? 32 : 16; }

template <int BM>
int sgemm_launch(hipStream_t st, const SgemmParams& p) {
  const dim3 grid((unsigned)(p.m / BM * (p.n / 64)), 1u, p.group_mode == JPP_GROUP_K ? (unsigned)p.n_seg : 1u);
  // (copies of 16 bytes, whole steps)
  const bool staged = BM <= 32 && !p.ta && !p.tb && p.k % 32 == 0 && (p.lda | p.ldb | p.stride_b) % 4 == 0 &&
                      ((uintptr_t)p.a | (uintptr_t)p.b) % 16 == 0;
  if constexpr (BM <= 32) {
    if (staged) {
      constexpr int SMEM = 4 * kStages32<BM> * (BM + 64) * 128;
      auto kern = sgemm_kernel<BM, false, false, true>;
      static std::once_flag configured;   // (the limit is sticky per kernel)
      static hipError_t configure_rc = hipSuccess;
      std::call_once(configured, [&] {
        configure_rc = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
      });
      JPP_CHECK_HIP(configure_rc);
      hipLaunchKernelGGL(kern, grid, dim3(256), SMEM, st, p);
      JPP_LAUNCH_CHECK();
      return JPP_OK;
    }
  }
  if (p.ta && p.tb) hipLaunchKernelGGL((sgemm_kernel<BM, true, true, false>), grid, dim3(256), 0, st, p);
  else if (p.ta) hipLaunchKernelGGL((sgemm_kernel<BM, true, false, false>), grid, dim3(256), 0, st, p);
  else if (p.tb) hipLaunchKernelGGL((sgemm_kernel<BM, false, true, false>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((sgemm_kernel<BM, false, false, false>), grid, dim3(256), 0, st, p);
  JPP_LAUNCH_CHECK();
  return JPP_OK;
}

// ---------------------------------------------------------------------------
// LayerNorm / RMSNorm: one wave per row
// ---------------------------------------------------------------------------
// N > 0: rows of at most 64 N columns, which a lane holds in registers, with its share of the scale and shift: one
// trip to memory instead of three loops of loads that wait for each other (512 x 256: 5.5 -> 3.2 us).
template <int N, bool COPY>
__global__ __launch_bounds__(256) void norm_fwd32_kernel(const float* __restrict__ x,
                                                         const float* __restrict__ gamma,
                                                         const float* __restrict__ beta,
                                                         float* __restrict__ y, float* mean_out,
                                                         float* rstd_out, long rows, int cols,
                                                         float eps, const float* __restrict__ copy_src,
                                                         float* __restrict__ copy_dst) {
// (the scaled and shifted value is three roundings in either form)
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float* xr = x + row * cols;
  float v[N ? N : 1], g[N ? N : 1], b[N ? N : 1];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int c = lane + 64 * i;
    const bool in = c < cols;
    v[i] = in ? xr[c] : 0.f;
    g[i] = in ? gamma[c] : 0.f;
    b[i] = in && beta ? beta[c] : 0.f;
  }
  if constexpr (COPY) {   // (as in the bf16 norm: the stage's input)
    if constexpr (N > 0) {
      float w[N];
#pragma unroll
      for (int i = 0; i < N; ++i) w[i] = lane + 64 * i < cols ? copy_src[row * cols + lane + 64 * i] : 0.f;
#pragma unroll
      for (int i = 0; i < N; ++i)
        if (lane + 64 * i < cols) copy_dst[row * cols + lane + 64 * i] = w[i];
    } else {
      for (int c = lane; c < cols; c += 64) copy_dst[row * cols + c] = copy_src[row * cols + c];
    }
  }
  float mean = 0.f;
  if (beta) {
    float s = 0.f;
    if constexpr (N > 0) {
#pragma unroll
      for (int i = 0; i < N; ++i) s += v[i];
    } else {
      for (int c = lane; c < cols; c += 64) s += xr[c];
    }
    mean = wave_sum(s) / cols;
  }
  float q = 0.f;
  if constexpr (N > 0) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const float d = lane + 64 * i < cols ? v[i] - mean : 0.f;
      q = __builtin_fmaf(d, d, q);
    }
  } else {
    for (int c = lane; c < cols; c += 64) {
      const float d = xr[c] - mean;
      q = __builtin_fmaf(d, d, q);
    }
  }
  const float rstd = rsqrtf(wave_sum(q) / cols + eps);
  auto scaled = [&](float x, float gamma) { return (x - mean) * rstd * gamma; };
  if constexpr (N > 0) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = lane + 64 * i;
      if (c < cols) y[row * cols + c] = beta ? scaled(v[i], g[i]) + b[i] : scaled(v[i], g[i]);
    }
  } else {
    for (int c = lane; c < cols; c += 64) {
      const float t = scaled(xr[c], gamma[c]);
      y[row * cols + c] = beta ? t + beta[c] : t;
    }
  }
  if (lane == 0) {
    if (mean_out) mean_out[row] = mean;
    rstd_out[row] = rstd;
  }
}

// Column sums of 16 adjacent columns over all rows by one workgroup of NT threads: 64 sums a column, sum rg
// over rows rg, rg + 64, ..., NT / 16 of them at a time; four adjacent ones meet first inside a wave, then the 16
// fours in order (whatever NT, the same sums).  These sums are latency and nothing
// else: one thread per column walks its rows one load after another, 4 to 16 waves on the whole
// device.  Spread like this a thread's loads are in flight together: the four bias gradients of
// a layer of hidden 256 on 512 tokens 4.8 us in one launch, a norm's backward 4.9 us.
struct ColSum {
  float a, b;
};
template <int NT, typename Load>
__device__ __forceinline__ ColSum column_sums(long rows, Load load) {
  __shared__ ColSum red[16][16];
  const int tid = threadIdx.x, c = tid & 15, wave = tid >> 6;
#pragma unroll 1
  for (int part = 0; part < 1024 / NT; ++part) {
    ColSum s = {0.f, 0.f};
    long r = (tid >> 4) + part * (NT / 16);
    for (; r + 7 * 64 < rows; r += 8 * 64) {
      ColSum v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = load(r + i * 64);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        s.a += v[i].a;
        s.b += v[i].b;
      }
    }
    for (; r < rows; r += 64) {
      const ColSum v = load(r);
      s.a += v.a;
      s.b += v.b;
    }
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {
      s.a += __shfl_xor(s.a, o);
      s.b += __shfl_xor(s.b, o);
    }
    if ((tid & 63) < 16) red[wave + part * (NT / 64)][c] = s;
  }
  __syncthreads();
  ColSum t = {0.f, 0.f};
  if (tid < 16)
    for (int w = 0; w < 16; ++w) {
      t.a += red[w][c].a;
      t.b += red[w][c].b;
    }
  return t;   // (threads 0 .. 15)
}

// Both halves of a norm's backward in one launch (they read the same tensors and neither reads
// what the other writes): the first `row_blocks` workgroups take 16 rows each, one wave per
// row, for dx; each of the others the parameter gradients of 16 columns,
// dgamma[c] += sum_r dy[r,c] xhat[r,c], dbeta[c] += sum_r dy[r,c].
__global__ __launch_bounds__(1024) void norm_bwd32_kernel(const float* __restrict__ dy,
                                                          const float* __restrict__ x,
                                                          const float* mean_in,
                                                          const float* __restrict__ rstd_in,
                                                          const float* __restrict__ gamma,
                                                          const float* resid, float* __restrict__ dx,
                                                          float* dgamma, float* dbeta, long rows,
                                                          int cols, int row_blocks) {
  if ((int)blockIdx.x >= row_blocks) {
    const int col = ((int)blockIdx.x - row_blocks) * 16 + (threadIdx.x & 15);
    const bool in = col < cols;
    const ColSum s = column_sums<1024>(in ? rows : 0, [&](long r) {
      const float d = dy[r * cols + col];
      const float mean = mean_in ? mean_in[r] : 0.f;
      return ColSum{d * (x[r * cols + col] - mean) * rstd_in[r], d};
    });
    if (threadIdx.x < 16 && in) {
      dgamma[col] += s.a;
      if (dbeta) dbeta[col] += s.b;
    }
    return;
  }
  const int lane = threadIdx.x & 63;
  const long row = (long)blockIdx.x * 16 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float rstd = rstd_in[row], mean = mean_in ? mean_in[row] : 0.f;
  const float* xr = x + row * cols;
  const float* dyr = dy + row * cols;
  float s1 = 0.f, s2 = 0.f;
  for (int c = lane; c < cols; c += 64) {
    const float dg = dyr[c] * gamma[c];
    s1 += dg;
    s2 += dg * (xr[c] - mean) * rstd;
  }
  s2 = wave_sum(s2) / cols;
  s1 = mean_in ? wave_sum(s1) / cols : 0.f;
  for (int c = lane; c < cols; c += 64) {
    const float xh = (xr[c] - mean) * rstd;
    float o = (dyr[c] * gamma[c] - s1 - xh * s2) * rstd;
    if (resid) o += resid[row * cols + c];
    dx[row * cols + c] = o;
  }
}

// acc[c] += sum_r x[r,c] of up to four matrices with the same rows; `first[i]`: first workgroup
// of matrix i (past the grid where there is none)
struct ColItems32 {
  const float* x[4];
  float* acc[4];
  long ld[4];
  int cols[4], first[4];
};
template <int NT>
__device__ __forceinline__ void colsum_block(const ColItems32& p, int blk, long rows) {
  const bool s1 = blk >= p.first[1], s2 = blk >= p.first[2], s3 = blk >= p.first[3];
#define JPP_PICK(field) (s3 ? p.field[3] : s2 ? p.field[2] : s1 ? p.field[1] : p.field[0])
  const float* const x = JPP_PICK(x);
  float* const acc = JPP_PICK(acc);
  const long ld = JPP_PICK(ld);
  const int cols = JPP_PICK(cols), col = (blk - JPP_PICK(first)) * 16 + (threadIdx.x & 15);
#undef JPP_PICK
  const bool in = col < cols;
  const ColSum s = column_sums<NT>(in ? rows : 0, [&](long r) { return ColSum{x[r * ld + col], 0.f}; });
  if (threadIdx.x < 16 && in) acc[col] += s.a;
}
__global__ __launch_bounds__(1024) void colsum32_kernel(ColItems32 p, long rows) {
  colsum_block<1024>(p, blockIdx.x, rows);
}

// A layer's weight gradients, up to four products C_i += A_i^T B_i over the same rows, and its bias gradients,
// column sums over them, in one launch: workgroups first[i] .. first[i + 1] - 1 take product i, those from
// col_first on the sums.  Apart, each fills a part of the device and is mostly latency: a layer of hidden 256 on
// 512 tokens 27 us in five launches, 17 as one and the sums'.  Which products gain by it: kWgrads32 below.
struct SgemmWgrads {
  SgemmParams p;        // what they share, and product 0
  const float* a[4];
  const float* b[4];
  float* c[4];
  long lda[4], ldb[4], ldc[4];
  int n[4], first[4], col_first;
  ColItems32 cols;
};
template <int BM>
__global__ __launch_bounds__(256) void sgemm_wgrads_kernel(SgemmWgrads w) {
  const int blk = blockIdx.x;
  if (blk >= w.col_first) {
    colsum_block<256>(w.cols, blk - w.col_first, w.p.k);
    return;
  }
  const bool s1 = blk >= w.first[1], s2 = blk >= w.first[2], s3 = blk >= w.first[3];
#define JPP_PICK(field) (s3 ? w.field[3] : s2 ? w.field[2] : s1 ? w.field[1] : w.field[0])
  SgemmParams p = w.p;
  p.a = JPP_PICK(a);
  p.b = JPP_PICK(b);
  p.c = JPP_PICK(c);
  p.lda = JPP_PICK(lda);
  p.ldb = JPP_PICK(ldb);
  p.ldc = JPP_PICK(ldc);
  p.n = JPP_PICK(n);
  const int first = JPP_PICK(first);
#undef JPP_PICK
  sgemm_tile<BM, true, true, false>(p, blk - first);
}

// loss = scale * mean((out - target)^2), dout = scale * 2 (out - target) / count: one
// workgroup, partial sums per thread in index order (eight elements' loads in flight), then a
// fixed tree
__global__ __launch_bounds__(1024) void mse32_kernel(const float* __restrict__ out,
                                                     const float* __restrict__ target, long count,
                                                     float scale, float* loss, float* dout) {
  __shared__ float red[1024];
  float s = 0.f;
  const float k = scale * 2.0f / (float)count;
  long i = threadIdx.x;
  for (; i + 7 * 1024 < count; i += 8 * 1024) {
    float d[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) d[e] = out[i + e * 1024] - target[i + e * 1024];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      s += d[e] * d[e];
      if (dout) dout[i + e * 1024] = k * d[e];
    }
  }
  for (; i < count; i += 1024) {
    const float d = out[i] - target[i];
    s += d * d;
    if (dout) dout[i] = k * d;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss[0] = scale * red[0] / (float)count;
}

// half-split rotary embedding in place on the first `heads` heads of each row
__global__ __launch_bounds__(256) void rope32_kernel(float* __restrict__ x, long ld,
                                                     const float* __restrict__ cos_tab,
                                                     const float* __restrict__ sin_tab, long rows,
                                                     int seq, int heads, int d, int inverse) {
  const int half = d / 2;
  const long total = rows * heads * half;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long)gridDim.x * 256) {
    const int j = (int)(i % half);
    const long th = i / half;
    const int hh = (int)(th % heads);
    const long t = th / heads;
    const int pos = (int)(t % seq);
    float* p = x + t * ld + hh * d + j;
    const float cs = cos_tab[(long)pos * half + j];
    const float sn = inverse ? -sin_tab[(long)pos * half + j] : sin_tab[(long)pos * half + j];
    const float a = p[0], b = p[half];
    p[0] = a * cs - b * sn;
    p[half] = b * cs + a * sn;
  }
}

// ---------------------------------------------------------------------------
// Attention on the fp32 matrix instruction, 16 rows of one side per workgroup: its waves take
// the other side's tiles of 16 rows in turn and meet in LDS, in wave order, at the end.  Sizes
// here are small (16 sequences and heads of 128 positions), so a workgroup per 16 rows and the
// split over its waves are what fills the device; operands go from L2 straight into MFMA
// fragments.  With c = lane % 16 and g = lane / 16, three layouts fit each other unchanged:
//   row fragment   row c, elements 16 t + 4 g .. + 3 of the head dimension: operand of a
//                  product over the head dimension
//   score tile     its result: row 4 g + r of the A side, row c of the B side in register r -
//                  which is the B operand of a product over the A side's rows
//   column frag.   row 4 g + r, elements 64 t + 4 c .. + 3: the A operand of that product; its
//                  result holds elements 64 t + 16 g + 4 r + j of row c (tile 4 t + j, register r)
// ---------------------------------------------------------------------------
struct Attn32 {
  const float *q, *k, *v, *d_o;
  float *o, *lse, *dq, *dk, *dv, *delta;
  long ldq, ldk, ldv, ldo, lddo, lddq, lddk, lddv;
  int batch, seq, n_heads, n_kv_heads, causal;
  float scale;
};

// (eight waves where their partial results and fragments have room, two per SIMD)
template <int D>
constexpr int kAttnWaves32 = D == 64 ? 8 : 4;

template <int D>
struct Rows32 {   // row fragments of 16 rows
  f32x4 v[D / 16];
  __device__ __forceinline__ void load(const float* p, long ld, int c, int g) {
#pragma unroll
    for (int t = 0; t < D / 16; ++t) v[t] = *(const f32x4_u*)(p + c * ld + 16 * t + 4 * g);
  }
};
template <int D>
struct Cols32 {   // column fragments of 16 rows
  f32x4 v[4][D / 64];
  __device__ __forceinline__ void load(const float* p, long ld, int c, int g) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int t = 0; t < D / 64; ++t) v[r][t] = *(const f32x4_u*)(p + (4 * g + r) * ld + 64 * t + 4 * c);
  }
};
// score tile of two sets of 16 rows
template <int D>
__device__ __forceinline__ f32x4 score32(const Rows32<D>& a, const Rows32<D>& b) {
  // two chains: an MFMA's result is the next one's input after 8 passes
  f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
  for (int t = 0; t < D / 16; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f32x4& s = e & 1 ? s1 : s0;
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[t][e], b.v[t][e], s, 0, 0, 0);
    }
  return s0 + s1;
}
// acc += (columns of the A side's 16 rows)^T (score tile)
template <int D>
__device__ __forceinline__ void outer32(f32x4 (&acc)[D / 16], const Cols32<D>& a, const f32x4& s) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int t = 0; t < D / 64; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[4 * t + j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[r][t][j], s[r], acc[4 * t + j], 0, 0, 0);
}
// sum and maximum over the four lanes that share c
__device__ __forceinline__ float quad_sum(float v) {
  v += __shfl_xor(v, 16);
  return v + __shfl_xor(v, 32);
}
__device__ __forceinline__ float quad_max(float v) {
  v = fmaxf(v, __shfl_xor(v, 16));
  return fmaxf(v, __shfl_xor(v, 32));
}
// The waves' accumulators, added in wave order, to 16 rows of `out`; `buf`: W x 16 x D floats of
// LDS that no wave reads any more.  Register r of tile 4 t + j, lane (c, g) is element
// 64 t + 16 g + 4 r + j of row c.
template <int D, int W>
__device__ __forceinline__ void store_sum32(const f32x4 (&acc)[D / 16], float* buf, float* out, long ld) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, g = lane >> 4;
#pragma unroll
  for (int t = 0; t < D / 64; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *(f32x4*)(buf + ((wave * (D / 64) + t) * 4 + r) * 256 + lane * 4) =
          f32x4{acc[4 * t][r], acc[4 * t + 1][r], acc[4 * t + 2][r], acc[4 * t + 3][r]};
  __syncthreads();
  // piece (t, r) of lane (c, g) is out[c][64 t + 16 g + 4 r ..]
  for (int i = tid; i < 16 * D / 4; i += 64 * W) {
    const int row = i / (D / 4), piece = i % (D / 4), t = piece / 16, pg = (piece >> 2) & 3, r = piece & 3;
    const float* src = buf + (t * 4 + r) * 256 + (pg * 16 + row) * 4;
    f32x4 v = *(const f32x4*)src;
#pragma unroll
    for (int w = 1; w < W; ++w) v += *(const f32x4*)(src + w * 16 * D);
    *(f32x4_u*)(out + row * ld + piece * 4) = v;
  }
}

template <int D>
__global__ __launch_bounds__(64 * kAttnWaves32<D>) void attn_fwd32_kernel(Attn32 p) {
  constexpr int W = kAttnWaves32<D>;
  __shared__ float buf[W * 16 * D];
  __shared__ float ms[W][16], ls[W][16];
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = blockIdx.y, b = blockIdx.z, hk = h / (p.n_heads / p.n_kv_heads);
  const int q0 = blockIdx.x * 16;
  const long row0 = (long)b * p.seq;
  Rows32<D> q;
  q.load(p.q + (row0 + q0) * p.ldq + h * D, p.ldq, c, g);
  f32x4 o[D / 16];
#pragma unroll
  for (int i = 0; i < D / 16; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const int kend = p.causal ? q0 + 16 : p.seq;
  const float* kp = p.k + row0 * p.ldk + hk * D;
  const float* vp = p.v + row0 * p.ldv + hk * D;
  for (int k0 = wave * 16; k0 < kend; k0 += W * 16) {
    Rows32<D> kr;
    Cols32<D> vc;
    kr.load(kp + k0 * p.ldk, p.ldk, c, g);
    vc.load(vp + k0 * p.ldv, p.ldv, c, g);
    f32x4 s = score32<D>(kr, q);
    float mx = m;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s[r] *= p.scale;
      if (p.causal && k0 + 4 * g + r > q0 + c) s[r] = -INFINITY;
      mx = fmaxf(mx, s[r]);
    }
    mx = quad_max(mx);
    // (a row whose scores so far are all -inf keeps a sum of zero)
    const float base = mx == -INFINITY ? 0.f : mx;
    const float alpha = expf(m - base);
    m = mx;
    l *= alpha;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s[r] = expf(s[r] - base);
      l += s[r];
    }
#pragma unroll
    for (int i = 0; i < D / 16; ++i) o[i] *= alpha;
    outer32<D>(o, vc, s);
  }
  l = quad_sum(l);
  if (g == 0) {
    ms[wave][c] = m;
    ls[wave][c] = l;
  }
  __syncthreads();
  float mall = ms[0][c];
#pragma unroll
  for (int w = 1; w < W; ++w) mall = fmaxf(mall, ms[w][c]);
  const float base = mall == -INFINITY ? 0.f : mall;
  float lall = 0.f;
#pragma unroll
  for (int w = 0; w < W; ++w) lall += ls[w][c] * expf(ms[w][c] - base);
  const float f = expf(m - base) / lall;
#pragma unroll
  for (int i = 0; i < D / 16; ++i) o[i] *= f;
  store_sum32<D, W>(o, buf, p.o + (row0 + q0) * p.ldo + h * D, p.ldo);
  if (threadIdx.x < 16) p.lse[((long)b * p.n_heads + h) * p.seq + q0 + c] = mall + logf(lall);
}

// this lane's share of delta = rowsum(dO o O) of row c, given the row's elements of dO
template <int D>
__device__ __forceinline__ float row_delta32(const Rows32<D>& go, const float* o_rows, long ldo, int c, int g) {
  Rows32<D> o;
  o.load(o_rows, ldo, c, g);
  float dl = 0.f;
#pragma unroll
  for (int t = 0; t < D / 16; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) dl = fmaf(go.v[t][e], o.v[t][e], dl);
  return quad_sum(dl);
}

// dQ of 16 queries, and delta for the dK/dV kernel behind it
template <int D>
__device__ __forceinline__ void dq_tile32(const Attn32& p, float* buf, int qt, int h, int b) {
  constexpr int W = kAttnWaves32<D>;
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hk = h / (p.n_heads / p.n_kv_heads);
  const int q0 = qt * 16;
  const long row0 = (long)b * p.seq;
  Rows32<D> q, go;
  q.load(p.q + (row0 + q0) * p.ldq + h * D, p.ldq, c, g);
  go.load(p.d_o + (row0 + q0) * p.lddo + h * D, p.lddo, c, g);
  const float dl = row_delta32<D>(go, p.o + (row0 + q0) * p.ldo + h * D, p.ldo, c, g);
  const long stat = ((long)b * p.n_heads + h) * p.seq + q0 + c;
  if (wave == 0 && g == 0) p.delta[stat] = dl;
  const float lse = p.lse[stat];
  f32x4 dq[D / 16];
#pragma unroll
  for (int i = 0; i < D / 16; ++i) dq[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int kend = p.causal ? q0 + 16 : p.seq;
  const float* kp = p.k + row0 * p.ldk + hk * D;
  const float* vp = p.v + row0 * p.ldv + hk * D;
  for (int k0 = wave * 16; k0 < kend; k0 += W * 16) {
    Rows32<D> kr, vr;
    Cols32<D> kc;
    kr.load(kp + k0 * p.ldk, p.ldk, c, g);
    vr.load(vp + k0 * p.ldv, p.ldv, c, g);
    kc.load(kp + k0 * p.ldk, p.ldk, c, g);
    f32x4 s = score32<D>(kr, q);
    const f32x4 dp = score32<D>(vr, go);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float pr = (p.causal && k0 + 4 * g + r > q0 + c) ? 0.f : expf(s[r] * p.scale - lse);
      s[r] = pr * (dp[r] - dl) * p.scale;
    }
    outer32<D>(dq, kc, s);
  }
  store_sum32<D, W>(dq, buf, p.dq + (row0 + q0) * p.lddq + h * D, p.lddq);
}

template <int D>
__global__ __launch_bounds__(64 * kAttnWaves32<D>) void attn_dq32_kernel(Attn32 p) {
  __shared__ float buf[kAttnWaves32<D> * 16 * D];
  dq_tile32<D>(p, buf, blockIdx.x, blockIdx.y, blockIdx.z);
}

// dK, dV of 16 keys: the waves take the 16-query tiles of every head of the keys' group in turn.  WITH_DQ: the whole
// backward in one launch (blockIdx.y: key heads, whose workgroups take longer, in front of the query heads).  delta is not
// there yet then and is formed here too (the same value).  (As a function that two kernels call, the registers
// of the one behind attn_dq32_kernel fall out worse: 7 heads of 128 on one key head, 2 x 640 rows under a mask 318 us, 305
// like this.)
template <int D, bool WITH_DQ>
__global__ __launch_bounds__(64 * kAttnWaves32<D>) void attn_dkv32_kernel(Attn32 p) {
  constexpr int W = kAttnWaves32<D>;
  __shared__ float buf[W * 16 * D];
  if constexpr (WITH_DQ) {
    if ((int)blockIdx.y >= p.n_kv_heads) {
      dq_tile32<D>(p, buf, blockIdx.x, blockIdx.y - p.n_kv_heads, blockIdx.z);
      return;
    }
  }
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hk = blockIdx.y, b = blockIdx.z, grp = p.n_heads / p.n_kv_heads;
  const int k0 = blockIdx.x * 16;
  const long row0 = (long)b * p.seq;
  Rows32<D> kr, vr;
  kr.load(p.k + (row0 + k0) * p.ldk + hk * D, p.ldk, c, g);
  vr.load(p.v + (row0 + k0) * p.ldv + hk * D, p.ldv, c, g);
  f32x4 dk[D / 16], dv[D / 16];
#pragma unroll
  for (int i = 0; i < D / 16; ++i) dk[i] = dv[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int first = p.causal ? k0 / 16 : 0, tiles = p.seq / 16 - first;
  for (int i = wave; i < grp * tiles; i += W) {
    const int h = hk * grp + i / tiles, q0 = (first + i % tiles) * 16;
    const float* qp = p.q + (row0 + q0) * p.ldq + h * D;
    const float* gp = p.d_o + (row0 + q0) * p.lddo + h * D;
    Rows32<D> qr, gr;
    Cols32<D> qc, gc;
    qr.load(qp, p.ldq, c, g);
    gr.load(gp, p.lddo, c, g);
    gc.load(gp, p.lddo, c, g);
    qc.load(qp, p.ldq, c, g);
    const long stat = ((long)b * p.n_heads + h) * p.seq + q0 + 4 * g;
    const f32x4 lse = *(const f32x4_u*)(p.lse + stat);
    f32x4 dl;
    if constexpr (WITH_DQ) {
      const float own = row_delta32<D>(gr, p.o + (row0 + q0) * p.ldo + h * D, p.ldo, c, g);
#pragma unroll
      for (int r = 0; r < 4; ++r) dl[r] = __shfl(own, 4 * g + r);
    } else {
      dl = *(const f32x4_u*)(p.delta + stat);
    }
    f32x4 s = score32<D>(qr, kr);
    const f32x4 dp = score32<D>(gr, vr);
    f32x4 ds;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s[r] = (p.causal && k0 + c > q0 + 4 * g + r) ? 0.f : expf(s[r] * p.scale - lse[r]);
      ds[r] = s[r] * (dp[r] - dl[r]) * p.scale;
    }
    outer32<D>(dv, gc, s);
    outer32<D>(dk, qc, ds);
  }
  store_sum32<D, W>(dv, buf, p.dv + (row0 + k0) * p.lddv + hk * D, p.lddv);
  __syncthreads();
  store_sum32<D, W>(dk, buf, p.dk + (row0 + k0) * p.lddk + hk * D, p.lddk);
}

// Whether a backward is one launch: while its workgroups are at most one per CU (its registers allow one).  Either
// half of a small one is a chain of latencies on part of the device, and they run beside each other in little more than
// the longer one's time (us, two launches / one: 4 heads x 64, 4 x 128 rows 16.9 / 9.2; 1 x 512 rows under a
// mask 34.3 / 19.1; 4 heads x 128, 4 x 128 rows 26.6 / 15.1); 384 and 512 workgroups 0.97 - 1.01 of the two's
// time, 1024 1.08.  One launch writes dQ, dK and dV while it reads everything else, where two read only
// part of it: a caller whose results lie over the inputs keeps the two.
constexpr long kBwdAtOnce = 256;
bool bwd32_at_once(const jpp_attn_args* a) {
  const int64_t rows = (int64_t)a->batch * a->seq;
  if (rows / 16 * (a->n_heads + a->n_kv_heads) > kBwdAtOnce) return false;
  struct Range {
    uintptr_t lo, hi;
  };
  auto range = [&](const void* p, int64_t ld, int heads) {
    return Range{(uintptr_t)p, (uintptr_t)p + (uintptr_t)(((rows - 1) * ld + heads * a->head_dim) * 4)};
  };
  const Range out[3] = {range(a->dq, a->lddq, a->n_heads), range(a->dk, a->lddk, a->n_kv_heads),
                        range(a->dv, a->lddv, a->n_kv_heads)};
  const Range in[6] = {range(a->q, a->ldq, a->n_heads), range(a->k, a->ldk, a->n_kv_heads),
                       range(a->v, a->ldv, a->n_kv_heads), range(a->o, a->ldo, a->n_heads),
                       range(a->d_o, a->lddo, a->n_heads),
                       {(uintptr_t)a->lse, (uintptr_t)a->lse + (uintptr_t)(rows * a->n_heads * 4)}};
  for (const Range& w : out)
    for (const Range& r : in)
      if (w.lo < r.hi && r.lo < w.hi) return false;
  return true;
}

int attn_check(const jpp_attn_args* a, const char* who, Attn32& p) {
  JPP_REQUIRE(a && a->q && a->k && a->v && a->o && a->lse, "%s: null operand", who);
  JPP_REQUIRE(a->head_dim == 64 || a->head_dim == 128, "%s: head_dim must be 64 or 128", who);
  JPP_REQUIRE(a->batch > 0 && a->seq > 0 && a->seq % 64 == 0, "%s: seq must be a multiple of 64", who);
  JPP_REQUIRE(a->n_heads > 0 && a->n_kv_heads > 0 && a->n_heads % a->n_kv_heads == 0,
              "%s: n_heads must be a multiple of n_kv_heads", who);
  JPP_REQUIRE(a->ldq >= (int64_t)a->n_heads * a->head_dim && a->ldo >= (int64_t)a->n_heads * a->head_dim &&
                  a->ldk >= (int64_t)a->n_kv_heads * a->head_dim &&
                  a->ldv >= (int64_t)a->n_kv_heads * a->head_dim,
              "%s: leading dimension too small", who);
  p.q = (const float*)a->q; p.k = (const float*)a->k; p.v = (const float*)a->v;
  p.o = (float*)a->o; p.lse = a->lse;
  p.d_o = (const float*)a->d_o; p.dq = (float*)a->dq; p.dk = (float*)a->dk; p.dv = (float*)a->dv;
  p.delta = a->delta;
  p.ldq = a->ldq; p.ldk = a->ldk; p.ldv = a->ldv; p.ldo = a->ldo;
  p.lddo = a->lddo; p.lddq = a->lddq; p.lddk = a->lddk; p.lddv = a->lddv;
  p.batch = a->batch; p.seq = a->seq; p.n_heads = a->n_heads; p.n_kv_heads = a->n_kv_heads;
  p.causal = a->causal;
  p.scale = 1.0f / sqrtf((float)a->head_dim);
  return JPP_OK;
}

}  // namespace

// Ways to run a layer's weight gradients: one launch on tiles of 16, 32 or 64 rows, or a launch per product (each on
// the tile that it takes by itself).  A CU takes one workgroup of any of them at a time.  Expected time, us, with
// w = rounds of the 256 CUs, s = tiles / 256, k = rows of the contraction / 1024:
//   w = 1   c0 + c1 k + s (c2 + c3 k)
//   w > 1   c0 + w (c1 + c2 k) + s (c3 + c4 k)
// (a round that all workgroups start together finds its operands in L2, later ones, out of step, do not: 512 x 2048
// outputs are one round and 38 us at 2048 rows, two such products and 192 tiles more in one grid 58 a round).
// Least squares of the relative error over 400 layers (hidden 64 .. 2048, feed-forward 1 .. 6 times that, 128 .. 8192
// rows, post- and pre-norm and gated ones, also without a feed-forward), mean error 1 - 6 %.  The smallest estimate takes 0.4 % over
// the best way, 9 % at worst; one launch always, on 64 rows from 512 strips of 16 on, 4 % and 82 %, and was slower than
// a launch per product by up to 37 % (hidden 512, feed-forward 2048, 4096 rows: 336 us, 269 apart).
struct Fit32 {
  float one[4], more[5];
};
constexpr Fit32 kWgrads32[2][3] = {
    {{{2.9f, 4.7f, 0.8f, 0.04f}, {0.f, 1.45f, 6.4f, 1.1f, 0.f}},     // a launch per product: 16, 32, 64 rows
     {{4.1f, 8.0f, 0.f, 0.f}, {0.f, 2.2f, 11.8f, 1.1f, 0.8f}},
     {{4.6f, 15.2f, 0.f, 0.f}, {5.7f, 0.f, 19.0f, 0.9f, 7.7f}}},
    {{{3.8f, 4.5f, 0.8f, 0.9f}, {3.6f, 0.35f, 5.95f, 0.8f, 1.2f}},   // one launch
     {{4.6f, 7.9f, 0.9f, 0.25f}, {3.9f, 1.35f, 9.0f, 0.3f, 5.4f}},
     {{4.5f, 15.0f, 0.95f, 0.25f}, {7.5f, 0.f, 18.7f, 0.4f, 8.7f}}}};

static float wgrads32_us(bool together, int rows, long strips, long contraction) {
  const int i = rows / 32;   // 16, 32, 64
  const Fit32& f = kWgrads32[together][i];
  const long tiles = strips >> i;
  const float k = contraction / 1024.f, s = tiles / 256.f, w = (float)((tiles + 255) / 256);
  return tiles <= 256 ? f.one[0] + f.one[1] * k + s * (f.one[2] + f.one[3] * k)
                      : f.more[0] + w * (f.more[1] + f.more[2] * k) + s * (f.more[3] + f.more[4] * k);
}

struct Wgrads32 {
  int rows;    // of a tile of the one launch; 0: a launch per product
  bool sums;   // the column sums go along
};

// The sums' workgroups cost next to nothing where they fit into the last round (0.05 of their own launch's time in the
// median).  Where they do not, each holds a CU for as long as its walk over all rows takes: behind a single round that
// is more than their own launch from 384 rows on (a layer of hidden 256 and 1024 on 512 tokens 18.8 us, 12.7 + 3.9
// apart; on 4096 122 and 66 + 15), among several rounds, whose tiles are out of step, from 1024 rows on (0.99 of the
// time up to there, 1.1 beyond).  Tiles of 16 rows leave room beside them: one round 0.7 - 0.9 up to 1024 rows, 1.17
// beyond, several 0.98.
static Wgrads32 wgrads32(int n, const jpp_gemm_args* g, int n_cols, const jpp_colsum_item* items) {
  long strips = 0;
  float best = 0.f;
  for (int i = 0; i < n; ++i) {
    const long own = (g[i].m / 16) * (g[i].n / 64);
    strips += own;
    best += wgrads32_us(false, tile_rows32(own), own, g[i].k);
  }
  Wgrads32 way = {0, false};
  for (int rows : {16, 32, 64}) {
    const float us = wgrads32_us(true, rows, strips, g[0].k);
    if (us < best) {
      best = us;
      way.rows = rows;
    }
  }
  if (!way.rows) return way;
  long tiles = 0, blocks = 0;
  for (int i = 0; i < n; ++i) tiles += (g[i].m / way.rows) * (g[i].n / 64);
  for (int i = 0; i < n_cols; ++i) blocks += (items[i].cols + 15) / 16;
  const long along = way.rows == 16 ? (tiles > 256 ? LONG_MAX : 1024) : tiles > 256 ? 768 : 256;   // rows
  way.sums = g[0].k <= along || (tiles + blocks + 255) / 256 == (tiles + 255) / 256;
  return way;
}

static int column_items(ColItems32& p, int n, const jpp_colsum_item* items) {
  int blocks = 0;
  for (int i = 0; i < 4; ++i) {
    const jpp_colsum_item& q = items[i < n ? i : 0];
    p.x[i] = (const float*)q.x;
    p.acc[i] = q.acc;
    p.ld[i] = q.ld;
    p.cols[i] = (int)q.cols;
    p.first[i] = i < n ? blocks : 0x7fffffff;
    if (i < n) blocks += (int)((q.cols + 15) / 16);
  }
  return blocks;
}

int jpp_colsum_f32_items(hipStream_t stream, int n, const jpp_colsum_item* items, int64_t rows) {
  JPP_REQUIRE(n >= 1 && n <= 4, "colsum_f32: 1 to 4 matrices");
  ColItems32 p;
  const int blocks = column_items(p, n, items);
  hipLaunchKernelGGL(colsum32_kernel, dim3((unsigned)blocks), dim3(1024), 0, stream, p, (long)rows);
  JPP_LAUNCH_CHECK();
  return JPP_OK;
}

int jpp_wgrads_f32(hipStream_t stream, int n, const jpp_gemm_args* g, int n_cols, const jpp_colsum_item* items) {
  JPP_REQUIRE(n >= 1 && n <= 4 && n_cols >= 0 && n_cols <= 4, "wgrads_f32: 1 to 4 products, up to 4 column sums");
  SgemmWgrads w;
  memset(&w, 0, sizeof(w));
  double flops = 0;
  for (int i = 0; i < 4; ++i) {
    const jpp_gemm_args& q = g[i < n ? i : 0];
    JPP_REQUIRE(q.k_parts <= 1 && q.k == g[0].k && q.k > 0 && q.k % 16 == 0 && q.m > 0 && q.m % 64 == 0 &&
                    q.n > 0 && q.n % 64 == 0 && q.lda >= q.m && q.ldb >= q.n && q.ldc >= q.n,
                "wgrads_f32: product %d has a shape of its own or a bad one", i);
    w.a[i] = (const float*)q.a; w.b[i] = (const float*)q.b; w.c[i] = (float*)q.c;
    w.lda[i] = q.lda; w.ldb[i] = q.ldb; w.ldc[i] = q.ldc; w.n[i] = (int)q.n;
    if (i < n) flops += 2.0 * q.m * q.n * q.k;
  }
  w.p.k = (int)g[0].k;
  w.p.ta = w.p.tb = 1;
  w.p.epi = JPP_EPI_ACC_F32;
  const Wgrads32 way = wgrads32(n, g, n_cols, items);
  if (!way.rows) {
    for (int i = 0; i < n; ++i)
      if (int rc = jpp_gemm_f32(stream, g + i)) return rc;
    return n_cols ? jpp_colsum_f32_items(stream, n_cols, items, g[0].k) : JPP_OK;
  }
  if (n_cols && !way.sums) {
    if (int rc = jpp_colsum_f32_items(stream, n_cols, items, g[0].k)) return rc;
    n_cols = 0;
  }
  const int bm = way.rows;
  int blocks = 0;
  for (int i = 0; i < 4; ++i) {
    w.first[i] = i < n ? blocks : 0x7fffffff;
    if (i < n) blocks += (int)(g[i].m / bm * (g[i].n / 64));
  }
  w.col_first = blocks;
  if (n_cols) blocks += column_items(w.cols, n_cols, items);
  ProbeScope probe(stream, n_cols ? "wgrads_f32_sums" : "wgrads_f32", flops, 0);
  if (bm == 64) hipLaunchKernelGGL(sgemm_wgrads_kernel<64>, dim3((unsigned)blocks), dim3(256), 0, stream, w);
  else if (bm == 32) hipLaunchKernelGGL(sgemm_wgrads_kernel<32>, dim3((unsigned)blocks), dim3(256), 0, stream, w);
  else hipLaunchKernelGGL(sgemm_wgrads_kernel<16>, dim3((unsigned)blocks), dim3(256), 0, stream, w);
  JPP_LAUNCH_CHECK();
  return JPP_OK;
}

int jpp_norm_fwd_copy_f32(hipStream_t stream, const jpp_norm_args* a, const void* copy_src, void* copy_dst) {
  JPP_REQUIRE(a && a->x && a->gamma && a->y && a->rstd, "norm_fwd_f32: null operand");
  JPP_REQUIRE(a->rows > 0 && a->cols > 0, "norm_fwd_f32: empty");
  JPP_REQUIRE((a->beta == nullptr) == (a->mean == nullptr),
              "norm_fwd_f32: beta and mean are both given (LayerNorm) or both NULL (RMSNorm)");
#define JPP_NF32(N) (copy_dst ? norm_fwd32_kernel<N, true> : norm_fwd32_kernel<N, false>)
  auto kern = a->cols <= 256 ? JPP_NF32(4) : a->cols <= 512 ? JPP_NF32(8) : a->cols <= 1024 ? JPP_NF32(16) : JPP_NF32(0);
#undef JPP_NF32
  hipLaunchKernelGGL(kern, dim3((unsigned)((a->rows + 3) / 4)), dim3(256), 0, stream, (const float*)a->x,
                     (const float*)a->gamma, (const float*)a->beta, (float*)a->y, a->mean, a->rstd, (long)a->rows,
                     (int)a->cols, a->eps, (const float*)copy_src, (float*)copy_dst);
  JPP_LAUNCH_CHECK();
  return JPP_OK;
}

extern "C" {

int jpp_gemm_f32(void* stream, const jpp_gemm_args* a) {
  JPP_REQUIRE(!a || a->k_parts <= 1, "gemm_f32: one operand pair per product");
  JPP_REQUIRE(a && a->a && a->b && a->c, "gemm_f32: null operand");
  JPP_REQUIRE(!a->rope_cos && !a->rope_sin,
              "gemm_f32: no rotary epilogue on f32 tensors (jpp_rope_f32 is the pass for them)");
  const bool group_k = a->group_mode == JPP_GROUP_K;
  JPP_REQUIRE(a->m > 0 && a->n > 0 && (a->k > 0 || group_k) && a->m % 64 == 0 && a->n % 64 == 0 &&
                  (a->k % 16 == 0 || group_k),
              "gemm_f32: M, N must be multiples of 64 and K of 16, got %ldx%ldx%ld", (long)a->m,
              (long)a->n, (long)a->k);
  if (a->group_mode != JPP_GROUP_NONE) {
    JPP_REQUIRE(a->group_mode == JPP_GROUP_M || group_k, "gemm_f32: unknown group_mode %d",
                a->group_mode);
    JPP_REQUIRE(a->seg && a->n_seg > 0 && a->n_seg <= 256, "gemm_f32: grouped problem needs seg[n_seg+1]");
    JPP_REQUIRE(!a->bias && !a->resid, "gemm_f32: grouped problems take no bias / residual");
    JPP_REQUIRE(!group_k || (a->trans_a && a->trans_b),
                "gemm_f32: a grouped contraction takes both operands with the rows as the slow index");
  }
  const int e = a->epilogue;
  JPP_REQUIRE(e >= JPP_EPI_BF16 && e <= JPP_EPI_DSWIGLU, "gemm_f32: unsupported epilogue %d", e);
  JPP_REQUIRE(a->lda >= (a->trans_a ? a->m : (group_k ? 0 : a->k)) &&
                  a->ldb >= (a->trans_b ? a->n : (group_k ? 0 : a->k)) && a->ldc >= a->n,
              "gemm_f32: leading dimension too small");
  if (e == JPP_EPI_GELU) JPP_REQUIRE(a->c2 && a->ldc2 >= a->n, "gemm_f32: GELU epilogue needs c2");
  if (e == JPP_EPI_DGELU) JPP_REQUIRE(a->aux && a->ldaux >= a->n, "gemm_f32: dGELU epilogue needs aux");
  if (e == JPP_EPI_SWIGLU)
    JPP_REQUIRE(a->c2 && a->ldc2 >= a->n / 2 && !a->bias && !a->resid,
                "gemm_f32: SwiGLU epilogue needs c2 [M, N/2] and takes no bias / residual");
  if (e == JPP_EPI_DSWIGLU)
    JPP_REQUIRE(a->aux && a->ldaux >= 2 * a->n && a->ldc >= 2 * a->n && !a->bias && !a->resid,
                "gemm_f32: dSwiGLU epilogue needs aux and C of width 2N and takes no bias / residual");
  if (a->resid) JPP_REQUIRE(a->ldresid >= a->n, "gemm_f32: bad ldresid");
  SgemmParams p;
  p.a = (const float*)a->a; p.b = (const float*)a->b; p.c = (float*)a->c; p.c2 = (float*)a->c2;
  p.bias = (const float*)a->bias; p.resid = (const float*)a->resid; p.aux = (const float*)a->aux;
  p.m = (int)a->m; p.n = (int)a->n; p.k = (int)a->k;
  p.lda = a->lda; p.ldb = a->ldb; p.ldc = a->ldc; p.ldc2 = a->ldc2; p.ldresid = a->ldresid;
  p.ldaux = a->ldaux;
  p.ta = a->trans_a != 0; p.tb = a->trans_b != 0; p.epi = e; p.gelu_tanh = a->gelu_tanh;
  p.seg = a->seg; p.n_seg = a->n_seg; p.group_mode = a->group_mode;
  p.stride_b = a->stride_b; p.stride_c = a->stride_c;
  const int rows = tile_rows32((a->m / 16) * (a->n / 64) * (group_k ? a->n_seg : 1));
  if (rows == 64) return sgemm_launch<64>((hipStream_t)stream, p);
  if (rows == 32) return sgemm_launch<32>((hipStream_t)stream, p);
  return sgemm_launch<16>((hipStream_t)stream, p);
}

int jpp_rope_f32(void* stream, float* x, int64_t ld, const float* cos_tab, const float* sin_tab,
                 int batch, int seq, int n_rot_heads, int head_dim, int inverse) {
  JPP_REQUIRE(x && cos_tab && sin_tab, "rope_f32: null operand");
  JPP_REQUIRE(batch > 0 && seq > 0 && n_rot_heads > 0 && head_dim > 0 && head_dim % 2 == 0 &&
                  ld >= (int64_t)n_rot_heads * head_dim,
              "rope_f32: bad shape");
  const long rows = (long)batch * seq, total = rows * n_rot_heads * (head_dim / 2);
  const unsigned grid = (unsigned)((total + 255) / 256 > 65536 ? 65536 : (total + 255) / 256);
  hipLaunchKernelGGL(rope32_kernel, dim3(grid), dim3(256), 0, (hipStream_t)stream, x, (long)ld,
                     cos_tab, sin_tab, rows, seq, n_rot_heads, head_dim, inverse);
  JPP_LAUNCH_CHECK();
  return JPP_OK;
}

int jpp_norm_fwd_f32(void* stream, const jpp_norm_args* a) {
  return jpp_norm_fwd_copy_f32((hipStream_t)stream, a, nullptr, nullptr);
}

int jpp_norm_bwd_f32(void* stream, const jpp_norm_args* a) {
  JPP_REQUIRE(a && a->x && a->gamma && a->dy && a->dx && a->rstd && a->dgamma,
              "norm_bwd_f32: null operand");
  JPP_REQUIRE(a->rows > 0 && a->cols > 0, "norm_bwd_f32: empty");
  JPP_REQUIRE(!a->mean || a->dbeta, "norm_bwd_f32: LayerNorm needs dbeta");
  hipStream_t st = (hipStream_t)stream;
  const unsigned row_blocks = (unsigned)((a->rows + 15) / 16), col_blocks = (unsigned)((a->cols + 15) / 16);
  hipLaunchKernelGGL(norm_bwd32_kernel, dim3(row_blocks + col_blocks), dim3(1024), 0, st,
                     (const float*)a->dy, (const float*)a->x, (const float*)a->mean,
                     (const float*)a->rstd, (const float*)a->gamma, (const float*)a->resid,
                     (float*)a->dx, a->dgamma, a->mean ? a->dbeta : nullptr, (long)a->rows,
                     (int)a->cols, (int)row_blocks);
  JPP_LAUNCH_CHECK();
  return JPP_OK;
}

int jpp_colsum_accum_f32(void* stream, const float* x, int64_t ld, int64_t rows, int64_t cols,
                         float* acc) {
  JPP_REQUIRE(x && acc && rows > 0 && cols > 0 && ld >= cols, "colsum_accum_f32: bad arguments");
  const jpp_colsum_item item = {x, ld, cols, acc};
  return jpp_colsum_f32_items((hipStream_t)stream, 1, &item, rows);
}

int jpp_mse_loss_f32(void* stream, const float* out, const float* target, int64_t count,
                     float scale, float* loss, float* dout) {
  JPP_REQUIRE(out && target && loss && count > 0, "mse_loss_f32: bad arguments");
  hipLaunchKernelGGL(mse32_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, out, target,
                     (long)count, scale, loss, dout);
  JPP_LAUNCH_CHECK();
  return JPP_OK;
}

int jpp_attn_fwd_f32(void* stream, const jpp_attn_args* a) {
  Attn32 p;
  if (int rc = attn_check(a, "attn_fwd_f32", p)) return rc;
  const dim3 grid((unsigned)(a->seq / 16), (unsigned)a->n_heads, (unsigned)a->batch);
  if (a->head_dim == 64)
    hipLaunchKernelGGL(attn_fwd32_kernel<64>, grid, dim3(64 * kAttnWaves32<64>), 0, (hipStream_t)stream, p);
  else
    hipLaunchKernelGGL(attn_fwd32_kernel<128>, grid, dim3(64 * kAttnWaves32<128>), 0, (hipStream_t)stream, p);
  JPP_LAUNCH_CHECK();
  return JPP_OK;
}

int jpp_attn_bwd_f32(void* stream, const jpp_attn_args* a) {
  Attn32 p;
  if (int rc = attn_check(a, "attn_bwd_f32", p)) return rc;
  JPP_REQUIRE(a->d_o && a->dq && a->dk && a->dv && a->delta, "attn_bwd_f32: null operand");
  JPP_REQUIRE(a->lddo >= (int64_t)a->n_heads * a->head_dim && a->lddq >= (int64_t)a->n_heads * a->head_dim &&
                  a->lddk >= (int64_t)a->n_kv_heads * a->head_dim &&
                  a->lddv >= (int64_t)a->n_kv_heads * a->head_dim,
              "attn_bwd_f32: leading dimension too small");
  hipStream_t st = (hipStream_t)stream;
  if (bwd32_at_once(a)) {
    const dim3 grid((unsigned)(a->seq / 16), (unsigned)(a->n_heads + a->n_kv_heads), (unsigned)a->batch);
    if (a->head_dim == 64) hipLaunchKernelGGL((attn_dkv32_kernel<64, true>), grid, dim3(64 * kAttnWaves32<64>), 0, st, p);
    else hipLaunchKernelGGL((attn_dkv32_kernel<128, true>), grid, dim3(64 * kAttnWaves32<128>), 0, st, p);
    JPP_LAUNCH_CHECK();
    return JPP_OK;
  }
  const dim3 gq((unsigned)(a->seq / 16), (unsigned)a->n_heads, (unsigned)a->batch);
  const dim3 gk((unsigned)(a->seq / 16), (unsigned)a->n_kv_heads, (unsigned)a->batch);
  if (a->head_dim == 64) {
    hipLaunchKernelGGL(attn_dq32_kernel<64>, gq, dim3(64 * kAttnWaves32<64>), 0, st, p);
    hipLaunchKernelGGL((attn_dkv32_kernel<64, false>), gk, dim3(64 * kAttnWaves32<64>), 0, st, p);
  } else {
    hipLaunchKernelGGL(attn_dq32_kernel<128>, gq, dim3(64 * kAttnWaves32<128>), 0, st, p);
    hipLaunchKernelGGL((attn_dkv32_kernel<128, false>), gk, dim3(64 * kAttnWaves32<128>), 0, st, p);
  }
  JPP_LAUNCH_CHECK();
  return JPP_OK;
}

}  // extern "C"
