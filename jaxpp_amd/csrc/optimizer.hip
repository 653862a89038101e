// The step on the far side of the microbatch loop: Adam on the f32 gradient accumulators
// the loop leaves behind (README.md:90-93 applies `optimizer.update` + `apply_updates` to
// the gradients `treduce` returns; examples/basic.py:234 uses `optax.adam`).  One pass over
// a flat tensor: reads gradient, both moments and the f32 weights, writes moments, weights
// and the bf16 copy the stage computes with, and can clear the accumulator for the next
// loop on the way - 16 bytes read and 18 written per parameter, all of it HBM traffic.
#include <math.h>

#include <algorithm>

#include "common.h"

namespace {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct AdamParams {
  float* grad;
  float* master;
  bf16_t* param;
  float* m;
  float* v;
  float lr, b1, b2, omb1, omb2, eps, bc1, bc2, gscale;  // omb = 1 - beta, bc = 1 - beta^t
  int zero_grad;
};

// the arithmetic of optax.adam (eps outside the root, eps_root = 0): m and v are the
// exponential averages of g and g^2, each divided by 1 - beta^t before use
__device__ __forceinline__ float adam_one(const AdamParams& p, float g, float w, float& m,
                                          float& v) {
  g *= p.gscale;
  m = p.b1 * m + p.omb1 * g;
  v = p.b2 * v + p.omb2 * g * g;
  const float mh = m / p.bc1, vh = v / p.bc2;
  return w - p.lr * mh / (sqrtf(vh) + p.eps);
}

template <bool CACHED, class T>
__device__ __forceinline__ T fetch(const T* p) {
  if constexpr (CACHED) return *p;
  else return __builtin_nontemporal_load(p);
}
template <bool CACHED, class T>
__device__ __forceinline__ void put(T v, T* p) {
  if constexpr (CACHED) *p = v;
  else __builtin_nontemporal_store(v, p);
}

// 8 parameters per lane: two 16-byte pieces of every f32 tensor, two of 8 bytes of the bf16, the second
// 64 pieces behind the first, so that every access of a wave is one run of memory.  Ten streams of HBM
// traffic and nothing else bound it.  One trip per wave: a grid that walks the tensors in strides has each
// workgroup in ten far-apart places at a time (4.96 TB/s at 6e8 parameters, 5.53 without).  184e6 parameters
// 1313 -> 1180 us, 6e8 4315 -> 3687.
// CACHED: through the caches, for tensors that the memory-side one may still hold from the gradients on (kCachedBytes).
// Larger ones go past them: nothing is read again before the next step.
template <bool MASTER, bool CACHED>
__global__ __launch_bounds__(256) void adam_kernel(AdamParams p, long n8) {
  const int lane = threadIdx.x & 63;
  const long waves = (long)gridDim.x * 4;
  // trip w: 128 pieces of four parameters (the last one's pieces may end before)
  for (long w = (long)blockIdx.x * 4 + (threadIdx.x >> 6); w * 64 < n8; w += waves) {
    const long at = w * 128 + lane, end = n8 * 2;
    f32x4 g[2], m[2], v[2], x[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const long i = at + 64 * u;
      if (i >= end) continue;
      g[u] = fetch<CACHED>((const f32x4*)p.grad + i);
      m[u] = fetch<CACHED>((const f32x4*)p.m + i);
      v[u] = fetch<CACHED>((const f32x4*)p.v + i);
      if (MASTER) {
        x[u] = fetch<CACHED>((const f32x4*)p.master + i);
      } else {
        const u32x2 q = fetch<CACHED>((const u32x2*)p.param + i);
        x[u] = f32x4{bf16lo_to_f32(q[0]), bf16hi_to_f32(q[0]), bf16lo_to_f32(q[1]), bf16hi_to_f32(q[1])};
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const long i = at + 64 * u;
      if (i >= end) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float me = m[u][e], ve = v[u][e];
        x[u][e] = adam_one(p, g[u][e], x[u][e], me, ve);
        m[u][e] = me;
        v[u][e] = ve;
      }
      put<CACHED>(m[u], (f32x4*)p.m + i);
      put<CACHED>(v[u], (f32x4*)p.v + i);
      if (MASTER) put<CACHED>(x[u], (f32x4*)p.master + i);
      if (p.param)
        put<CACHED>(u32x2{pack_bf16x2(x[u][0], x[u][1]), pack_bf16x2(x[u][2], x[u][3])},
                                    (u32x2*)p.param + i);
      if (p.zero_grad) put<CACHED>(f32x4{0.f, 0.f, 0.f, 0.f}, (f32x4*)p.grad + i);
    }
  }
}

template <bool MASTER>
__global__ void adam_tail_kernel(AdamParams p, long start, long count) {
  const long i = start + threadIdx.x;
  if (i >= count) return;
  float m = p.m[i], v = p.v[i];
  const float w = adam_one(p, p.grad[i], MASTER ? p.master[i] : bf16_to_f32(p.param[i]), m, v);
  p.m[i] = m;
  p.v[i] = v;
  if (MASTER) p.master[i] = w;
  if (p.param) p.param[i] = f32_to_bf16(w);
  if (p.zero_grad) p.grad[i] = 0.f;
}

// Bytes of all tensors of a step up to which it goes through the caches: three quarters of the memory-side one.  8.4e6
// parameters (151 MB) again and again 38 us, past the caches 45; with 64 MB of other traffic between 39 and 48, with
// 512 MB 60 and 49.  Rows with the step at their end (activations, weights and gradients between): 3.5e6 parameters
// 607 us and 615, 7.1e6 699 and 710, 9.8e6 (177 MB) 3717 and 3720; 12.6e6 (227 MB) 3211 and 3157, 14.2e6 1821 and 1804.
constexpr int64_t kCachedBytes = 192 << 20;

}  // namespace

extern "C" int jpp_adam_step(void* stream, const jpp_adam_args* a) {
  JPP_REQUIRE(a && a->grad && a->m && a->v && (a->master || a->param),
              "adam_step: null operand (grad, m, v and one of master / param are required)");
  JPP_REQUIRE(a->count >= 0, "adam_step: negative count");
  JPP_REQUIRE(((uintptr_t)a->grad | (uintptr_t)a->m | (uintptr_t)a->v | (uintptr_t)a->master |
               (uintptr_t)a->param) % 16 == 0,
              "adam_step: operands must be 16-byte aligned");
  JPP_REQUIRE(a->step >= 1, "adam_step: step counts from 1, got %ld", (long)a->step);
  JPP_REQUIRE(a->beta1 >= 0. && a->beta1 < 1. && a->beta2 >= 0. && a->beta2 < 1.,
              "adam_step: beta1, beta2 must lie in [0, 1)");
  if (a->count == 0) return JPP_OK;
  AdamParams p;
  p.grad = a->grad; p.master = a->master; p.param = (bf16_t*)a->param; p.m = a->m; p.v = a->v;
  // every scalar is formed in double and rounded once, as a Python float that meets an f32
  // array is
  p.lr = (float)a->lr; p.b1 = (float)a->beta1; p.b2 = (float)a->beta2; p.eps = (float)a->eps;
  p.omb1 = (float)(1.0 - a->beta1);
  p.omb2 = (float)(1.0 - a->beta2);
  p.bc1 = (float)(1.0 - pow(a->beta1, (double)a->step));
  p.bc2 = (float)(1.0 - pow(a->beta2, (double)a->step));
  p.gscale = (float)a->grad_scale;
  p.zero_grad = a->zero_grad;
  hipStream_t st = (hipStream_t)stream;
  const double bytes = 12.0 + 8.0 + (a->master ? 8.0 : 2.0) + (a->param ? 2.0 : 0.0) +
                       (a->zero_grad ? 4.0 : 0.0);
  const bool cached = a->count * (12 + (a->master ? 4 : 0) + (a->param ? 2 : 0)) <= kCachedBytes;
  ProbeScope probe(st, "adam", 0, bytes * a->count);
  ProbeScope form(st, cached ? "adam_cached" : "adam_streamed", 0, bytes * a->count);   // (for a probe of one form alone)
  const long n8 = a->count / 8;
  const int grid = (int)std::min<long>(std::max<long>((n8 + 255) / 256, 1), 1 << 23);   // (2^31 threads)
  if (n8) {
    auto kern = a->master ? (cached ? adam_kernel<true, true> : adam_kernel<true, false>)
                          : (cached ? adam_kernel<false, true> : adam_kernel<false, false>);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, st, p, n8);
  }
  if (a->count % 8) {
    if (a->master)
      hipLaunchKernelGGL(adam_tail_kernel<true>, dim3(1), dim3(8), 0, st, p, n8 * 8, (long)a->count);
    else
      hipLaunchKernelGGL(adam_tail_kernel<false>, dim3(1), dim3(8), 0, st, p, n8 * 8, (long)a->count);
  }
  JPP_LAUNCH_CHECK();
  return JPP_OK;
}
