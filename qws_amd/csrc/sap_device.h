// sap_device.h -- what the fused SAP kernels share, whatever the block shape.
#pragma once

#include "kernels.h"
#include "sap.h"

namespace qws {

// y = A x for the packed Hermitian 6x6 whose reals k sit in a(k)
template <typename A>
__device__ __forceinline__ void herm6_mult_f(A a, const Cx<float> x[6], Cx<float> y[6]) {
#pragma unroll
  for (int r = 0; r < 6; ++r) y[r] = cscale(a(r), x[r]);
  int p = 6;
#pragma unroll
  for (int r = 0; r < 6; ++r)
#pragma unroll
    for (int c = r + 1; c < 6; ++c) {
      Cx<float> m = {a(p), a(p + 1)};
      y[r] = cfma(m, x[c], y[r]);
      y[c] = cfmac(m, x[r], y[c]);
      p += 2;
    }
}

// The site's clover inverse held in registers for the whole launch: 72 FP32 reals,
// or for FP16 storage 36 packed pairs (converted to FP32 at each use).
template <typename S> struct CloverRegs;
template <> struct CloverRegs<float> {
  float c[72];
  __device__ __forceinline__ void load(const float* C, long long s, long long V) {
    CloverIO<float>::load_chir<true>(C, s, V, 0, c);
    CloverIO<float>::load_chir<true>(C, s, V, 1, c + 36);
  }
  __device__ __forceinline__ float get(int k) const { return c[k]; }
};
template <> struct CloverRegs<__half> {
  __half2 c[36];
  __device__ __forceinline__ void load(const __half* C, long long s, long long V) {
    const Half4* p = reinterpret_cast<const Half4*>(C);
#pragma unroll
    for (int f = 0; f < 18; ++f) {
      const Half4 h = p[(long long)f * V + s];
      c[2 * f] = h.a;
      c[2 * f + 1] = h.b;
    }
  }
  __device__ __forceinline__ float get(int k) const {
    const float2 f = __half22float2(c[k >> 1]);
    return (k & 1) ? f.y : f.x;
  }
};

template <typename S>
__device__ __forceinline__ void clover_regs(const CloverRegs<S>& cl, Cx<float> v[12]) {
  Cx<float> x[6], y0[6], y1[6];
#pragma unroll
  for (int c = 0; c < 3; ++c) { x[c] = cadd(v[c * 4 + 0], v[c * 4 + 2]); x[3 + c] = cadd(v[c * 4 + 1], v[c * 4 + 3]); }
  herm6_mult_f([&](int k) { return cl.get(k); }, x, y0);
#pragma unroll
  for (int c = 0; c < 3; ++c) { x[c] = csub(v[c * 4 + 0], v[c * 4 + 2]); x[3 + c] = csub(v[c * 4 + 1], v[c * 4 + 3]); }
  herm6_mult_f([&](int k) { return cl.get(36 + k); }, x, y1);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    v[c * 4 + 0] = cadd(y0[c], y1[c]);
    v[c * 4 + 2] = csub(y0[c], y1[c]);
    v[c * 4 + 1] = cadd(y0[3 + c], y1[3 + c]);
    v[c * 4 + 3] = csub(y0[3 + c], y1[3 + c]);
  }
}

// BiCGStab's direction update folded into the first sweep (SAP_SRC_PUPD):
// p_c = r_c + beta (p_c - omega q_c) for this site, stored back to p, which the sweep
// then reads as its source.
__device__ __forceinline__ void src_update(const SapSrcUpdate& u, int r, long long off, long long site, long long V) {
  const Scalars& sc = u.sc[r];
  const float wr = (float)sc.omega[0], wi = (float)sc.omega[1], br = (float)sc.beta[0], bi = (float)sc.beta[1];
  float4* P = reinterpret_cast<float4*>(u.p + off);
  const float4* Q = reinterpret_cast<const float4*>(u.q + off);
  const float4* R = reinterpret_cast<const float4*>(u.r + off);
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    float4 pv = P[j * V + site];
    const float4 qv = Q[j * V + site], rv = R[j * V + site];
    bicg_p_update<float>(pv.x, pv.y, qv.x, qv.y, rv.x, rv.y, wr, wi, br, bi);
    bicg_p_update<float>(pv.z, pv.w, qv.z, qv.w, rv.z, rv.w, wr, wi, br, bi);
    P[j * V + site] = pv;
  }
}

}  // namespace qws
