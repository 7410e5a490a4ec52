// Pooling as the kernels share it: its own launch (llattn_pool.hip) and the one that also casts the weights
// (llattn_cast.hip).
#pragma once

#include <algorithm>

#include "llattn_abi.h"
#include "llattn_device.h"

namespace llattn {

struct PoolArgs {  // backward: x is dpooled (rows indexed by segment), out is dx (rows indexed by token)
  const void* x; int64_t x_sb, x_st;
  void* out; int64_t o_sb, o_sn;
  int B, T, D, seg, n_seg, divisor, accumulate;
};

__device__ __forceinline__ float seg_scale(int n, const PoolArgs& a) {
  if (a.divisor == LLATTN_DIV_COUNT) return 1.f / (float)(min((n + 1) * a.seg, a.T) - n * a.seg);
  if (a.divisor == LLATTN_DIV_SEG) return 1.f / (float)a.seg;
  return 1.f;
}

template <typename T>
__device__ __forceinline__ void load_vec16(const T* p, float (&v)[Vec16<T>::N]) {
  const uint4 x = ld16(p);
  const T* e = reinterpret_cast<const T*>(&x);
#pragma unroll
  for (int j = 0; j < Vec16<T>::N; ++j) v[j] = to_f<T>(e[j]);
}
template <typename T>
__device__ __forceinline__ void store_vec16(T* p, const float (&v)[Vec16<T>::N]) {
  uint4 x;
  T* e = reinterpret_cast<T*>(&x);
#pragma unroll
  for (int j = 0; j < Vec16<T>::N; ++j) e[j] = from_f<T>(v[j]);
  st16(p, x);
}

constexpr int kPoolLds = 8 * 32 * 8;  // floats of LDS of one workgroup (bf16 rows; half of it for fp32)

// One workgroup of 256: segment `seg` (of all batches) and column strip `strip` of 32 x 16 bytes.
template <typename T>
__device__ __forceinline__ void pool_strip(const PoolArgs& a, int seg, int strip, float* lds) {
  constexpr int V = Vec16<T>::N;
  float(*red)[32 * V] = reinterpret_cast<float(*)[32 * V]>(lds);
  const int n = seg % a.n_seg, b = seg / a.n_seg;
  const int cthr = threadIdx.x & 31, rg = threadIdx.x >> 5;
  const int col = (strip * 32 + cthr) * V;
  const int t0 = n * a.seg, t1 = min(t0 + a.seg, a.T);
  float acc[V];
#pragma unroll
  for (int j = 0; j < V; ++j) acc[j] = 0.f;
  if (col < a.D) {
    const T* xb = static_cast<const T*>(a.x) + b * a.x_sb + col;
    int t = t0 + rg;
    for (; t + 24 < t1; t += 32) {  // four rows in flight, added in the same order as one by one
      float v[4][V];
#pragma unroll
      for (int i = 0; i < 4; ++i) load_vec16<T>(xb + (int64_t)(t + 8 * i) * a.x_st, v[i]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < V; ++j) acc[j] += v[i][j];
    }
    for (; t < t1; t += 8) {
      float v[V];
      load_vec16<T>(xb + (int64_t)t * a.x_st, v);
#pragma unroll
      for (int j = 0; j < V; ++j) acc[j] += v[j];
    }
  }
#pragma unroll
  for (int j = 0; j < V; ++j) red[rg][cthr * V + j] = acc[j];
  __syncthreads();
  if (rg == 0 && col < a.D) {
    const float sc = seg_scale(n, a);
    float v[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
      float s = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) s += red[k][cthr * V + j];
      v[j] = s * sc;
    }
    store_vec16<T>(static_cast<T*>(a.out) + b * a.o_sb + (int64_t)n * a.o_sn + col, v);
  }
}

// workgroups of a pooling along (segments, column strips)
inline dim3 pool_grid(const PoolArgs& a, int dtype) {
  const int V = 16 / (int)elem_size(dtype);
  return dim3(a.B * a.n_seg, (a.D + 32 * V - 1) / (32 * V));
}

// Checks a pooling (forward: x, out; backward: dpooled, dx).  llattn_pool.hip.
int32_t check_pool(const char* who, const PoolArgs& a, int32_t dtype);

// Weight casts and poolings of one step in one launch; the arguments of llattn_cast_transposed and the poolings'.
// llattn_cast.hip.
constexpr int kCastPools = 2;
int32_t cast_and_pool(int32_t nseg, const float* const* src, void* const* dst, const int64_t* n,
                      const int32_t* dst_dtype, void* const* dst_t, const int64_t* ld_t, const int32_t* rows,
                      const PoolArgs* pools, int32_t n_pools, int32_t pool_dtype, void* stream);

}  // namespace llattn
