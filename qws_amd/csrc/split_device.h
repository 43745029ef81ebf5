// split_device.h -- what the operators with four waves per 64 sites share (split.hip, eo.hip).
#pragma once

#include "kernels.h"

namespace qws {
namespace split {

constexpr int SITES = 64;  // per workgroup of 4 waves

// The element of plane k (V sites each) at byte offset `at` of the plane: a uniform
// address and a 32-bit lane offset, no 64-bit address per load in vector registers.
template <typename T> __device__ __forceinline__ T get(const void* base, long long k, long long V, unsigned at) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + k * V * (long long)sizeof(T) + at);
}
template <typename T> __device__ __forceinline__ void put(void* base, long long k, long long V, unsigned at, T x) {
  *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + k * V * (long long)sizeof(T) + at) = x;
}

// FP32 and FP16 storage: planes of four reals; FP64: planes of two
template <typename S> struct IO {
  static constexpr unsigned Q = 4 * sizeof(S);  // bytes per site of a spinor or clover plane
  static __device__ __forceinline__ float4 quad(const S* p, int k, long long V, unsigned at) {
    if constexpr (sizeof(S) == 4) {
      return get<float4>(p, k, V, at);
    } else {
      const Half4 h = get<Half4>(p, k, V, at);
      const float2 x = __half22float2(h.a), y = __half22float2(h.b);
      return make_float4(x.x, x.y, y.x, y.y);
    }
  }
  // components 2j, 2j + 1
  static __device__ __forceinline__ void load2(const S* p, int j, long long V, unsigned at, Cx<float> v[2]) {
    const float4 q = quad(p, j, V, at);
    v[0] = {q.x, q.y}, v[1] = {q.z, q.w};
  }
  static __device__ __forceinline__ void store2(S* p, int j, long long V, unsigned at, const Cx<float> v[2]) {
    if constexpr (sizeof(S) == 4) {
      put(p, j, V, at, make_float4(v[0].re, v[0].im, v[1].re, v[1].im));
    } else {
      Half4 h;
      h.a = __floats2half2_rn(v[0].re, v[0].im);
      h.b = __floats2half2_rn(v[1].re, v[1].im);
      put(p, j, V, at, h);
    }
  }
  static __device__ __forceinline__ Cx<float> link(const S* U, int k, long long V, unsigned at) {
    if constexpr (sizeof(S) == 4) {
      const float2 q = get<float2>(U, k, V, at);
      return {q.x, q.y};
    } else {
      const float2 q = __half22float2(get<__half2>(U, k, V, at));
      return {q.x, q.y};
    }
  }
  static __device__ __forceinline__ void chir(const S* C, int i, long long V, unsigned at, float a[36]) {
#pragma unroll
    for (int f = 0; f < 9; ++f) {
      const float4 q = quad(C, 9 * i + f, V, at);
      a[4 * f] = q.x, a[4 * f + 1] = q.y, a[4 * f + 2] = q.z, a[4 * f + 3] = q.w;
    }
  }
};
template <> struct IO<double> {
  static constexpr unsigned Q = 16;
  static __device__ __forceinline__ Cx<double> link(const double* p, int k, long long V, unsigned at) {
    const double2 q = get<double2>(p, k, V, at);
    return {q.x, q.y};
  }
  static __device__ __forceinline__ void load2(const double* p, int j, long long V, unsigned at, Cx<double> v[2]) {
    v[0] = link(p, 2 * j, V, at), v[1] = link(p, 2 * j + 1, V, at);
  }
  static __device__ __forceinline__ void store2(double* p, int j, long long V, unsigned at, const Cx<double> v[2]) {
    put(p, 2 * j, V, at, make_double2(v[0].re, v[0].im));
    put(p, 2 * j + 1, V, at, make_double2(v[1].re, v[1].im));
  }
  static __device__ __forceinline__ void chir(const double* C, int i, long long V, unsigned at, double a[36]) {
#pragma unroll
    for (int f = 0; f < 18; ++f) {
      const Cx<double> q = link(C, 18 * i + f, V, at);
      a[2 * f] = q.re, a[2 * f + 1] = q.im;
    }
  }
};
template <typename S> constexpr unsigned LINK_BYTES = 2 * sizeof(S);

// rows 3H .. 3H+2 of herm6_mult, each summed in its order
template <int H, typename R>
__device__ __forceinline__ void herm3_mult(const R a[36], const Cx<R> x[6], Cx<R> y[3]) {
#pragma unroll
  for (int k = 0; k < 3; ++k) y[k] = cscale(a[3 * H + k], x[3 * H + k]);
  int p = 6;
#pragma unroll
  for (int r = 0; r < 6; ++r)
#pragma unroll
    for (int c = r + 1; c < 6; ++c) {
      const Cx<R> m = {a[p], a[p + 1]};
      if (r / 3 == H) y[r - 3 * H] = cfma(m, x[c], y[r - 3 * H]);
      if (c / 3 == H) y[c - 3 * H] = cfmac(m, x[r], y[c - 3 * H]);
      p += 2;
    }
}

}  // namespace split
}  // namespace qws
