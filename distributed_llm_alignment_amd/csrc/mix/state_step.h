// One token's update of a head's fp32 state [vdim, dim] (kept transposed), shared by the decode steps of retention and
// gated linear attention: S <- a o S + k v^T, o = S q, for dim % 4 == 0, dim <= 4 LPR.
//
// A workgroup of 512 owns (sequence, head) or a share of its value rows; LPR lanes hold a row, four channels
// each, a group of lanes eight consecutive rows. Bound by latency for few (sequence, head) pairs and by the state's
// bytes, read and written once, for many. So the first 8 rows a lane owns (a whole 128 x 128 state) are on their way
// before anything else is loaded, q, k and v go straight to the lanes that use them (no LDS, no barrier
// before the update), the row sums fold the eight rows and the lanes together (9 exchanges for 32 lanes instead of
// 40), and one barrier separates the update from the norm, which every wave forms for itself. The state passes the
// caches by: the other layers' states and weights come before its next use (32 rows x 16 heads of 128 x 128, in a
// replayed graph: 15.8 us against 18.9 with cached accesses).
#pragma once
#include "mma.h"

namespace dla {

constexpr int kStepThreads = 512, kStepRows = 8;

template <int LPR>
__device__ __forceinline__ void step_load(const float* S, int r0, int vhi, int dim, bool fresh, f32x4 (&s)[kStepRows]) {
  const int i = 4 * (threadIdx.x % LPR);
#pragma unroll
  for (int u = 0; u < kStepRows; ++u) {
    s[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (r0 + u < vhi && i < dim && !fresh) s[u] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(S + static_cast<int64_t>(r0 + u) * dim + i));
  }
}

// acc[u] summed over a group's LPR >= 8 lanes; a lane returns row (lane's top three bits)'s sum
template <int LPR>
__device__ __forceinline__ float step_reduce(const float (&acc)[kStepRows]) {
  const int li = threadIdx.x % LPR;
  const bool u4 = li & LPR / 2, u2 = li & LPR / 4, u1 = li & LPR / 8;
  float a[4], b[2];
#pragma unroll
  for (int j = 0; j < 4; ++j) a[j] = (u4 ? acc[j + 4] : acc[j]) + __shfl_xor(u4 ? acc[j] : acc[j + 4], LPR / 2, 64);
#pragma unroll
  for (int j = 0; j < 2; ++j) b[j] = (u2 ? a[j + 2] : a[j]) + __shfl_xor(u2 ? a[j] : a[j + 2], LPR / 4, 64);
  float v = (u1 ? b[1] : b[0]) + __shfl_xor(u1 ? b[0] : b[1], LPR / 8, 64);
#pragma unroll
  for (int o = LPR / 16; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Rows vlo .. vhi - 1: `s` holds the first pass's rows (step_load at vlo + 8 group). `value(r, v)`: v of rows r .. r + 7.
// Outputs go to `put(row, sum)`.
template <int LPR, typename Value, typename Put>
__device__ __forceinline__ void step_rows(float* S, int vlo, int vhi, int dim, bool fresh, f32x4 q, f32x4 k, f32x4 a,
                                          f32x4 (&s)[kStepRows], Value value, Put put) {
  constexpr int NG = kStepThreads / LPR;
  const int li = threadIdx.x % LPR, i = 4 * li;
  for (int r0 = vlo + kStepRows * (threadIdx.x / LPR); r0 < vhi; r0 += kStepRows * NG) {
    float v[kStepRows], acc[kStepRows];
    value(r0, v);
    f32x4 next[kStepRows];
    const bool more = r0 + kStepRows * NG < vhi;
    if (more) step_load<LPR>(S, r0 + kStepRows * NG, vhi, dim, fresh, next);
#pragma unroll
    for (int u = 0; u < kStepRows; ++u) {
      acc[u] = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[u][e] = a[e] * s[u][e] + k[e] * v[u];
        acc[u] += s[u][e] * q[e];
      }
      if (r0 + u < vhi && i < dim) __builtin_nontemporal_store(s[u], reinterpret_cast<f32x4*>(S + static_cast<int64_t>(r0 + u) * dim + i));
    }
    const float sum = step_reduce<LPR>(acc);
    const int row = r0 + li / (LPR / 8);
    if (li % (LPR / 8) == 0 && row < vhi) put(row, sum);
    if (more) {
#pragma unroll
      for (int u = 0; u < kStepRows; ++u) s[u] = next[u];
    }
  }
}

// v of rows r .. r + 7 of a projected row, zero past vdim or in padding
template <typename T>
__device__ __forceinline__ void step_values(const T* in, int r, int vdim, bool vec, bool pad, float (&v)[kStepRows]) {
  if (vec) {
    load_vec<T, kStepRows>(in + r, v);
#pragma unroll
    for (int u = 0; u < kStepRows; ++u) v[u] = pad ? 0.f : v[u];
  } else {
#pragma unroll
    for (int u = 0; u < kStepRows; ++u) v[u] = r + u < vdim && !pad ? to_f<T>(in[r + u]) : 0.f;
  }
}

// A share of the value rows is done: whether this workgroup was the last of a pair's `n` and so finishes it. The outputs
// were stored with device scope; `cnt` is zero before and after.
__device__ __forceinline__ bool step_last(int* cnt, int n) {
  __shared__ int last;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    last = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
    if (last) {
      __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
  }
  __syncthreads();
  return last;
}

// 1 / rms of o[0 .. n), formed by every wave
__device__ __forceinline__ float step_rstd(const float* o, int n, float eps) {
  float ss = 0.f;
  for (int v = threadIdx.x & 63; v < n; v += 64) ss += o[v] * o[v];
  return rsqrtf(wave_sum(ss) / n + eps);
}

}  // namespace dla
