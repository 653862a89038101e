// Attention for problems that do not fill the device with blocks of 128 queries or 64 keys.
//
// A workgroup owns 16 rows of one head's queries (keys, for dK / dV) and its eight waves take
// the other side 32 rows at a time in turn; their partial results meet in LDS, in wave order,
// at the end (deterministic, no atomics).  That reads the other side once per 16 rows instead of once per
// 64 to 256, which a large problem cannot afford and a small one does not notice: here a kernel's time is
// how long one workgroup takes, and it takes an eighth of the steps.
//
// Every wave copies the 32 rows of its next step into LDS of its own, whole lines in flight under the
// products of this one, and waits for nothing else: no barrier before the waves meet (but the forward's, which
// share a row's maximum).  Row fragments are plain reads of that tile, column fragments transposing ones.
// (Fragments loaded from memory directly take 16 rows x 64 bytes an instruction, which holds the CU's path
// several times as long as its kilobyte, and the rows of both products once each: backward of 16 heads x 512 x 64
// 35.3 us that way, 21.1 like this; of 16 and 4 heads x 512 x 128 without a mask 60 and 33; forward of 8 heads x 1024 x
// 64 16.2 and 11.0.)  What is left of a step is latency: the copies of one tile cannot start before the
// last fragment of the one before is out of it.  Tried: the rows of the output that dK / dV's row sums need a step
// ahead in registers (0 - 8 % slower).
//
// With c = lane % 16 and g = lane / 16 the layouts fit each other unchanged
// (v_mfma_f32_16x16x32_bf16: lane supplies row c, contraction elements 8 g .. 8 g + 7; a result
// register r is row 4 g + r of the A side, row c of the B side):
//   row fragment   row c, elements 32 t + 8 g .. + 7 of the head: a product over the head
//   score tiles    two results (u = 0, 1), rows 16 u + 4 g + r of the A side: rounded to bf16,
//                  their eight values are the B operand of a product over those 32 rows, whose
//                  contraction element 8 g + 4 u + r is row 16 u + 4 g + r
//   column frag.   tile j: element 16 j + c of rows 16 u + 4 g + r, two transposing reads of four rows
#include "attention_common.h"

using namespace jpp_attn;

namespace {

constexpr int W = 8;   // waves: two per SIMD

// row fragments of 16 rows
template <int D>
struct Rows {
  bf16x8 v[D / 32];
  __device__ __forceinline__ void load(const bf16_t* p, long ld, int c, int g) {
#pragma unroll
    for (int t = 0; t < D / 32; ++t) v[t] = *(const bf16x8*)(p + c * ld + 32 * t + 8 * g);
  }
  // of rows row0 .. row0 + 15 of a tile in LDS
  __device__ __forceinline__ void read(const uint8_t* tile, int row0, int c, int g) {
#pragma unroll
    for (int t = 0; t < D / 32; ++t) v[t] = *(const bf16x8*)(tile + (t >> 1) * 4096 + slab_off(row0 + c, (t & 1) * 4 + g));
  }
};

// column fragments of a tile in LDS
template <int D>
struct Cols {
  bf16x8 v[D / 16];
  __device__ __forceinline__ void read(const uint8_t* tile, int c, int g) {
#pragma unroll
    for (int j = 0; j < D / 16; ++j) {
      const int n = 16 * j + ((c & 3) << 2);
      const uint8_t* p = tile + (n >> 6) * 4096 + slab_off(4 * g + (c >> 2), (n & 63) >> 3) + ((n & 7) << 1);
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)JPP_LDS_PTR(p));
      const s16x4 hi =
          __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)JPP_LDS_PTR(p + 16 * 128));
      v[j] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  }
};

// A wave's copies of 32 rows of a head (D / 64 slabs of [32][64]) into a tile of LDS of its own.
template <int D>
struct TileCopy {
  using Slab = DmaTile<32, false, 1>;
  static constexpr int BYTES = 32 * D * 2, COPIES = D / 64 * Slab::INSTS;
  typename Slab::Offsets off;
  __device__ __forceinline__ TileCopy(long ld, int lane) { Slab::offsets(off, ld, 0, lane); }
  __device__ __forceinline__ void issue(const bf16_t* src, uint32_t tile) const {
#pragma unroll
    for (int q = 0; q < D / 64; ++q) Slab::template issue<0, Slab::INSTS>(uniform_ptr(src + 64 * q), off, tile + q * 4096, 0);
  }
};

template <int D>
__device__ __forceinline__ f32x4 score(const Rows<D>& a, const Rows<D>& b) {
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < D / 32; ++t) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v[t], b.v[t], s, 0, 0, 0);
  return s;
}

// acc += (columns of 32 rows)^T (their two score tiles)
template <int D>
__device__ __forceinline__ void outer(f32x4 (&acc)[D / 16], const Cols<D>& a, const f32x4 (&s)[2]) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const u32x4 q = {pack2(s[0][0], s[0][1]), pack2(s[0][2], s[0][3]), pack2(s[1][0], s[1][1]),
                   pack2(s[1][2], s[1][3])};
  const bf16x8 b = __builtin_bit_cast(bf16x8, q);
#pragma unroll
  for (int j = 0; j < D / 16; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v[j], b, acc[j], 0, 0, 0);
}

__device__ __forceinline__ float quad_sum(float v) {   // over the four lanes that share c
  v += __shfl_xor(v, 16);
  return v + __shfl_xor(v, 32);
}

template <int D>
__device__ __forceinline__ void clear(f32x4 (&acc)[D / 16]) {
#pragma unroll
  for (int j = 0; j < D / 16; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// The waves' accumulators, added in wave order and scaled, to 16 rows of `out` in bf16; with
// tables they leave rotated back (element d pairs with d + D/2; rounded to bf16 first, as a
// separate pass would read them back from memory), row i being position pos0 + i.  Register r
// of tile j, lane (c, g) is element 16 j + 4 g + r of row c.  `buf`: W x 16 x D floats of LDS.
template <int D>
__device__ __forceinline__ void store_sum(const f32x4 (&acc)[D / 16], float* buf, bf16_t* out, long ld,
                                          float scale, const float* cos_tab, const float* sin_tab, int pos0) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  __syncthreads();   // (the waves' tiles, or what was summed before, lie there)
#pragma unroll
  for (int j = 0; j < D / 16; ++j) *(f32x4*)(buf + (wave * (D / 16) + j) * 256 + lane * 4) = acc[j];
  __syncthreads();
  // quad k of a row: elements 4 k .. 4 k + 3
  auto quad = [&](int row, int k) {
    const float* src = buf + (k * 16 + row) * 4;
    f32x4 v = *(const f32x4*)src;
#pragma unroll
    for (int w = 1; w < W; ++w) v += *(const f32x4*)(src + w * 16 * D);
    return v;
  };
  if (tid < 16 * D / 8) {
    const int row = tid / (D / 8), k = tid % (D / 8);
    f32x4 a = quad(row, k), b = quad(row, k + D / 8);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      a[e] *= scale;
      b[e] *= scale;
    }
    if (cos_tab) {
      const f32x4 cs = *(const f32x4*)(cos_tab + (long)(pos0 + row) * (D / 2) + 4 * k);
      const f32x4 sn = *(const f32x4*)(sin_tab + (long)(pos0 + row) * (D / 2) + 4 * k);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = (float)(__bf16)a[e], y = (float)(__bf16)b[e];
        a[e] = x * cs[e] + y * sn[e];
        b[e] = y * cs[e] - x * sn[e];
      }
    }
    bf16_t* dst = out + row * ld + 4 * k;
    *(uint2*)dst = make_uint2(pack2(a[0], a[1]), pack2(a[2], a[3]));
    *(uint2*)(dst + D / 2) = make_uint2(pack2(b[0], b[1]), pack2(b[2], b[3]));
  }
}

// 16 queries of one head
template <int D, bool CAUSAL>
__global__ __launch_bounds__(64 * W) void attn_small_fwd_kernel(AttnParams p) {
  extern __shared__ __align__(16) float buf[];
  __shared__ float ms[2][W][16], ls[W][16];
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = blockIdx.x, b = blockIdx.z, hk = h / (p.n_heads / p.n_kv_heads);
  const int q0 = (CAUSAL ? gridDim.y - 1 - blockIdx.y : blockIdx.y) * 16;   // heavy blocks first
  const long row0 = (long)b * p.seq;
  Rows<D> q;
  q.load(p.q + (row0 + q0) * p.ldq + h * D, p.ldq, c, g);
  f32x4 o[D / 16];
  clear<D>(o);
  float m = -INFINITY, l = 0.f;
  const float sc = p.scale * kLog2e;
  const int kend = CAUSAL ? q0 + 16 : p.seq;
  const bf16_t* kp = p.k + row0 * p.ldk + hk * D;
  const bf16_t* vp = p.v + row0 * p.ldv + hk * D;
  using Copy = TileCopy<D>;
  const Copy ck(p.ldk, lane), cv(p.ldv, lane);
  const uint8_t* const kt = (const uint8_t*)buf + wave * (2 * Copy::BYTES);
  const uint8_t* const vt = kt + Copy::BYTES;
  if (wave * 32 < kend) {
    ck.issue(kp + (long)(wave * 32) * p.ldk, lds_address(kt));
    cv.issue(vp + (long)(wave * 32) * p.ldv, lds_address(vt));
  }
  // Rounds of W x 32 keys.  The waves share the running maximum: the probabilities are rounded
  // to bf16 for the second product, and against a reference other than the row's maximum they
  // round differently from a plain softmax's.
  int par = 0;
  for (int r0 = 0; r0 < kend; r0 += W * 32, par ^= 1) {
    const int k0 = r0 + wave * 32, kn = k0 + W * 32;
    const bool live = k0 < kend;   // (wave-uniform)
    f32x4 s[2];
    float mx = -INFINITY;
    if (live) {
      Rows<D> kr[2];
      dma_wait<Copy::COPIES>();    // K is in (copies land in order)
      kr[0].read(kt, 0, c, g);
      kr[1].read(kt, 16, c, g);
      lds_wait_all();
      if (kn < kend) ck.issue(kp + (long)kn * p.ldk, lds_address(kt));
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        s[u] = score<D>(kr[u], q);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (CAUSAL && k0 + 16 * u + 4 * g + r > q0 + c) s[u][r] = -INFINITY;
          mx = fmaxf(mx, s[u][r]);
        }
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
    }
    if (g == 0) ms[par][wave][c] = mx;
    __syncthreads();   // (one a round: the next round's maxima go to the other half)
    float m_new = m;
#pragma unroll
    for (int w = 0; w < W; ++w) m_new = fmaxf(m_new, ms[par][w][c]);
    const float neg = -m_new * sc;
    if (r0 > 0) {
      const float alpha = fast_exp2(fmaf(m, sc, neg));
      l *= alpha;
#pragma unroll
      for (int j = 0; j < D / 16; ++j) o[j] *= alpha;
    }
    m = m_new;
    if (live) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[u][r] = fast_exp2(fmaf(s[u][r], sc, neg));
          l += s[u][r];
        }
      Cols<D> vc;
      if (kn < kend) dma_wait<Copy::COPIES>();   // V is in; the next keys may be on their way
      else dma_wait_all();
      vc.read(vt, c, g);
      lds_wait_all();
      if (kn < kend) cv.issue(vp + (long)kn * p.ldv, lds_address(vt));
      outer<D>(o, vc, s);
    }
  }
  l = quad_sum(l);
  if (g == 0) ls[wave][c] = l;
  __syncthreads();
  float lall = 0.f;
#pragma unroll
  for (int w = 0; w < W; ++w) lall += ls[w][c];
  const float inv = 1.0f / lall;
#pragma unroll
  for (int j = 0; j < D / 16; ++j) o[j] *= inv;
  store_sum<D>(o, buf, p.o + (row0 + q0) * p.ldo + h * D, p.ldo, 1.0f, nullptr, nullptr, 0);
  if (threadIdx.x < 16) p.lse[((long)b * p.n_heads + h) * p.seq + q0 + c] = m * p.scale + logf(lall);
}

// sum over the head of dO * O, for row c
template <int D>
__device__ __forceinline__ float row_delta(const Rows<D>& d_o, const bf16_t* o, long ld, int c, int g) {
  Rows<D> of;
  of.load(o, ld, c, g);
  float acc = 0.f;
#pragma unroll
  for (int t = 0; t < D / 32; ++t)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc = fmaf((float)d_o.v[t][e], (float)of.v[t][e], acc);
  return quad_sum(acc);
}

// The whole backward as one launch: the first kv_blocks workgroups dK / dV of 16 keys each (the
// queries of every head of the key's group), the others dQ of 16 queries; both form the row
// term delta = sum dO * O themselves.
template <int D, bool CAUSAL>
__global__ __launch_bounds__(64 * W) void attn_small_bwd_kernel(AttnParams p, int kv_blocks) {
  extern __shared__ __align__(16) float buf[];
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = p.n_heads / p.n_kv_heads, tiles = p.seq / 16;
  const float sc = p.scale * kLog2e;
  if ((int)blockIdx.x < kv_blocks) {
    // (kv head fastest, then the tile - under a mask the first keys see the most queries)
    const int hk = blockIdx.x % p.n_kv_heads, rest = blockIdx.x / p.n_kv_heads;
    const int b = rest % p.batch, k0 = rest / p.batch * 16;
    const long row0 = (long)b * p.seq;
    Rows<D> kr, vr;
    kr.load(p.k + (row0 + k0) * p.ldk + hk * D, p.ldk, c, g);
    vr.load(p.v + (row0 + k0) * p.ldv + hk * D, p.ldv, c, g);
    f32x4 dk[D / 16], dv[D / 16];
    clear<D>(dk);
    clear<D>(dv);
    const int first = CAUSAL ? k0 / 32 : 0, steps = p.seq / 32 - first;
    using Copy = TileCopy<D>;
    const Copy cq(p.ldq, lane), cg(p.lddo, lane);
    const uint8_t* const qt = (const uint8_t*)buf + wave * (2 * Copy::BYTES);
    const uint8_t* const gt = qt + Copy::BYTES;
    auto copy = [&](int i) {
      const int h = hk * grp + i / steps, q0 = (first + i % steps) * 32;
      cq.issue(p.q + (row0 + q0) * p.ldq + h * D, lds_address(qt));
      cg.issue(p.d_o + (row0 + q0) * p.lddo + h * D, lds_address(gt));
    };
    if (wave < grp * steps) copy(wave);
    for (int i = wave; i < grp * steps; i += W) {
      const int h = hk * grp + i / steps, q0 = (first + i % steps) * 32;
      const bf16_t* op = p.o + (row0 + q0) * p.ldo + h * D;
      const float* lp = p.lse + ((long)b * p.n_heads + h) * p.seq + q0 + 4 * g;
      f32x4 s[2], ds[2];
      dma_wait_all();
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        Rows<D> qr, gr;
        qr.read(qt, 16 * u, c, g);
        gr.read(gt, 16 * u, c, g);
        const f32x4 lse = *(const f32x4*)(lp + 16 * u);
        const float dl = row_delta<D>(gr, op + 16 * u * p.ldo, p.ldo, c, g);
        s[u] = score<D>(qr, kr);
        ds[u] = score<D>(gr, vr);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float pr = fast_exp2(fmaf(s[u][r], sc, -lse[r] * kLog2e));
          if (CAUSAL && k0 + c > q0 + 16 * u + 4 * g + r) pr = 0.f;
          s[u][r] = pr;
          ds[u][r] = pr * (ds[u][r] - __shfl(dl, 4 * g + r));
        }
      }
      Cols<D> qc, gc;
      gc.read(gt, c, g);
      qc.read(qt, c, g);
      lds_wait_all();
      if (i + W < grp * steps) copy(i + W);
      outer<D>(dv, gc, s);
      outer<D>(dk, qc, ds);
    }
    store_sum<D>(dv, buf, p.dv + (row0 + k0) * p.lddv + hk * D, p.lddv, 1.0f, nullptr, nullptr, 0);
    store_sum<D>(dk, buf, p.dk + (row0 + k0) * p.lddk + hk * D, p.lddk, p.scale, p.rope_cos, p.rope_sin, k0);
    return;
  }
  const int blk = blockIdx.x - kv_blocks, h = blk % p.n_heads, rest = blk / p.n_heads;
  const int b = rest % p.batch, tile = rest / p.batch, hk = h / grp;
  const int q0 = (CAUSAL ? tiles - 1 - tile : tile) * 16;
  const long row0 = (long)b * p.seq;
  Rows<D> q, go;
  q.load(p.q + (row0 + q0) * p.ldq + h * D, p.ldq, c, g);
  go.load(p.d_o + (row0 + q0) * p.lddo + h * D, p.lddo, c, g);
  const float lse2 = p.lse[((long)b * p.n_heads + h) * p.seq + q0 + c] * kLog2e;
  const float dl = row_delta<D>(go, p.o + (row0 + q0) * p.ldo + h * D, p.ldo, c, g);
  f32x4 dq[D / 16];
  clear<D>(dq);
  const int kend = CAUSAL ? q0 + 16 : p.seq;
  const bf16_t* kp = p.k + row0 * p.ldk + hk * D;
  const bf16_t* vp = p.v + row0 * p.ldv + hk * D;
  using Copy = TileCopy<D>;
  const Copy ck(p.ldk, lane), cv(p.ldv, lane);
  const uint8_t* const kt = (const uint8_t*)buf + wave * (2 * Copy::BYTES);
  const uint8_t* const vt = kt + Copy::BYTES;
  auto copy = [&](int k0) {
    ck.issue(kp + (long)k0 * p.ldk, lds_address(kt));
    cv.issue(vp + (long)k0 * p.ldv, lds_address(vt));
  };
  if (wave * 32 < kend) copy(wave * 32);
  for (int k0 = wave * 32; k0 < kend; k0 += W * 32) {
    dma_wait_all();
    f32x4 ds[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      Rows<D> kr, vr;
      kr.read(kt, 16 * u, c, g);
      vr.read(vt, 16 * u, c, g);
      const f32x4 s = score<D>(kr, q), dp = score<D>(vr, go);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float pr = fast_exp2(fmaf(s[r], sc, -lse2));
        if (CAUSAL && k0 + 16 * u + 4 * g + r > q0 + c) pr = 0.f;
        ds[u][r] = pr * (dp[r] - dl);
      }
    }
    Cols<D> kc;
    kc.read(kt, c, g);
    lds_wait_all();
    if (k0 + W * 32 < kend) copy(k0 + W * 32);
    outer<D>(dq, kc, ds);
  }
  store_sum<D>(dq, buf, p.dq + (row0 + q0) * p.lddq + h * D, p.lddq, p.scale, p.rope_cos, p.rope_sin, q0);
}

// a tile of either operand per wave, over them the sums of 16 rows
template <int D>
constexpr int small_smem() {
  return W * 2 * TileCopy<D>::BYTES;
}
static_assert(small_smem<64>() >= W * 16 * 64 * 4 && small_smem<128>() >= W * 16 * 128 * 4, "room for the sums");

template <int D, bool CAUSAL>
int fwd(hipStream_t st, const AttnParams& p) {
  if (int rc = set_smem(attn_small_fwd_kernel<D, CAUSAL>, small_smem<D>())) return rc;
  hipLaunchKernelGGL((attn_small_fwd_kernel<D, CAUSAL>),
                     dim3((unsigned)p.n_heads, (unsigned)(p.seq / 16), (unsigned)p.batch), dim3(64 * W),
                     small_smem<D>(), st, p);
  JPP_LAUNCH_CHECK();
  return JPP_OK;
}

template <int D, bool CAUSAL>
int bwd(hipStream_t st, const AttnParams& p) {
  const int kv = p.seq / 16 * p.n_kv_heads * p.batch, q = p.seq / 16 * p.n_heads * p.batch;
  if (int rc = set_smem(attn_small_bwd_kernel<D, CAUSAL>, small_smem<D>())) return rc;
  hipLaunchKernelGGL((attn_small_bwd_kernel<D, CAUSAL>), dim3((unsigned)(kv + q)), dim3(64 * W),
                     small_smem<D>(), st, p, kv);
  JPP_LAUNCH_CHECK();
  return JPP_OK;
}

}  // namespace

namespace jpp_attn {

int launch_small_fwd(hipStream_t st, const AttnParams& p, int head_dim, bool causal) {
  if (head_dim == 64) return causal ? fwd<64, true>(st, p) : fwd<64, false>(st, p);
  return causal ? fwd<128, true>(st, p) : fwd<128, false>(st, p);
}

int launch_small_bwd(hipStream_t st, const AttnParams& p, int head_dim, bool causal) {
  if (head_dim == 64) return causal ? bwd<64, true>(st, p) : bwd<64, false>(st, p);
  return causal ? bwd<128, true>(st, p) : bwd<128, false>(st, p);
}

}  // namespace jpp_attn
