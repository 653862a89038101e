// Column sums of bf16 matrices of few rows by one workgroup per 64 columns, without partial sums in memory: a
// launch of their own (elementwise.hip), or workgroups beside the weight gradients of the same rows (gemm.hip).
#pragma once
#include <type_traits>
#include "common.h"

// Sums over `rows` of load(r, a, b), which adds 8 columns of row r into a (and b), for 64
// adjacent columns; thread t < 64 returns column t's two sums.  A thread owns 8 columns of every (NT PASSES / 8)-th
// row, in PASSES passes; the row groups of a column meet inside a wave first, then in order (NT PASSES decides
// the sums).  `red`: NT PASSES / 64 rows of LDS.
template <int NT, int UNROLL, int PASSES, class Load>
__device__ __forceinline__ float2 column_sums64(long rows, float2 (*red)[64], Load load) {
  constexpr int G = NT * PASSES / 8;
  const int tid = threadIdx.x;
#pragma unroll 1
  for (int pass = 0; pass < PASSES; ++pass) {
    float a[8], b[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] = b[e] = 0.f;
    long r = (tid >> 3) + pass * (NT / 8);
    for (; r + (UNROLL - 1) * G < rows; r += UNROLL * G) load(r, G, std::integral_constant<int, UNROLL>{}, a, b);
    for (; r < rows; r += G) load(r, G, std::integral_constant<int, 1>{}, a, b);
#pragma unroll
    for (int o = 8; o < 64; o <<= 1)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        a[e] += __shfl_xor(a[e], o);
        b[e] += __shfl_xor(b[e], o);
      }
    if ((tid & 63) < 8)
#pragma unroll
      for (int e = 0; e < 8; ++e) red[(tid >> 6) + pass * (NT / 64)][(tid & 7) * 8 + e] = make_float2(a[e], b[e]);
  }
  __syncthreads();
  float2 t = make_float2(0.f, 0.f);
  if (tid < 64)
#pragma unroll
    for (int w = 0; w < NT * PASSES / 64; ++w) {
      t.x += red[w][tid].x;
      t.y += red[w][tid].y;
    }
  return t;
}

// the bias gradients of a layer: workgroups first[i] .. first[i + 1] - 1 take tensor i
struct ColsumPanels {
  const bf16_t* x[4];
  long ld[4];
  float* acc[4];
  int cols[4], first[4];
};

// one of their workgroups, of NT threads; `red`: 16 rows of LDS
template <int NT>
__device__ __forceinline__ void colsum_panel(const ColsumPanels& p, int blk, long rows, float2 (*red)[64]) {
  const bool s1 = blk >= p.first[1], s2 = blk >= p.first[2], s3 = blk >= p.first[3];
#define JPP_PICK(f) (s3 ? f[3] : s2 ? f[2] : s1 ? f[1] : f[0])
  const bf16_t* const x = JPP_PICK(p.x);
  const long ld = JPP_PICK(p.ld);
  float* const acc = JPP_PICK(p.acc);
  const int c0 = (blk - JPP_PICK(p.first)) * 64, cols = JPP_PICK(p.cols);
#undef JPP_PICK
  const int c = c0 + (threadIdx.x & 7) * 8;
  const bf16_t* src = x + c;
  const float2 t = column_sums64<NT, 8, 1024 / NT>(
      c < cols ? rows : 0, red, [&](long r, int g, auto u, float (&a)[8], float (&)[8]) {
        constexpr int U = decltype(u)::value;
        uint4 v[U];
#pragma unroll
        for (int i = 0; i < U; ++i) v[i] = *(const uint4*)(src + (r + i * g) * ld);
#pragma unroll
        for (int i = 0; i < U; ++i) {
          float f[8];
          unpack8(v[i], f);
#pragma unroll
          for (int e = 0; e < 8; ++e) a[e] += f[e];
        }
      });
  if (threadIdx.x < 64 && c0 + (int)threadIdx.x < cols) acc[c0 + threadIdx.x] += t.x;
}

// Checks the tensors and lays out their workgroups; how many those are, or 0 where `rows` are too many.
int colsum_panels(int n, const jpp_colsum_item* items, int64_t rows, ColsumPanels* p, int* blocks);
