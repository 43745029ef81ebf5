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

// ---- FP16 operands with FP32 accumulation: the link and clover products use
// v_dot2_f32_f16 (two FP16 products summed into an FP32 accumulator), the spin
// projections packed FP16 adds, the hop sums, the clover results and the iterate
// update FP32.
typedef _Float16 h2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ h2v swp(h2v a) { return __builtin_shufflevector(a, a, 1, 0); }
__device__ __forceinline__ h2v neg_hi(h2v a) { return h2v{a.x, -a.y}; }
// c + a.x b.x + a.y b.y (v_dot2_f32_f16).  Only the compiler's own dot instructions
// are used, so that its hazard checks see every dependent pair.
__device__ __forceinline__ float dot2(h2v a, h2v b, float c) { return __builtin_amdgcn_fdot2(a, b, c, false); }
__device__ __forceinline__ h2v to_h2(Cx<float> v) { return h2v{(_Float16)v.re, (_Float16)v.im}; }
__device__ __forceinline__ Cx<float> from_h2(h2v v) { return {(float)v.x, (float)v.y}; }

// FP16 spin projection of the hop along MU, DIR (the table of project<>, packed)
template <int MU, int DIR>
__device__ __forceinline__ void project_h2(const h2v v[12], h2v a[6]) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const h2v s0 = v[c * 4 + 0], s1 = v[c * 4 + 1], s2 = v[c * 4 + 2], s3 = v[c * 4 + 3];
    h2v a0, a1;
    // i z = (-z.y, z.x), -i z = (z.y, -z.x)
    if (MU == 0) {
      if (DIR > 0) { a0 = s0 + h2v{s3.y, -s3.x}; a1 = s1 + h2v{s2.y, -s2.x}; }
      else         { a0 = s0 + h2v{-s3.y, s3.x}; a1 = s1 + h2v{-s2.y, s2.x}; }
    } else if (MU == 1) {
      if (DIR > 0) { a0 = s0 - s3; a1 = s1 + s2; } else { a0 = s0 + s3; a1 = s1 - s2; }
    } else if (MU == 2) {
      if (DIR > 0) { a0 = s0 + h2v{s2.y, -s2.x}; a1 = s1 + h2v{-s3.y, s3.x}; }
      else         { a0 = s0 + h2v{-s2.y, s2.x}; a1 = s1 + h2v{s3.y, -s3.x}; }
    } else {
      if (DIR > 0) { a0 = s2; a1 = s3; } else { a0 = s0; a1 = s1; }
    }
    a[c * 2 + 0] = a0;
    a[c * 2 + 1] = a1;
  }
}

// b = W a (forward) or W^+ a (backward), W[i][j] = c[j][i] as in link_mult<>.
// With A = (a.x, a.y): u a = (u.A', u.As), A' = (a.x, -a.y), As = (a.y, a.x);
// conj(u) a = (u.A, u.As'), As' = (a.y, -a.x).
template <int DIR>
__device__ __forceinline__ void link_mult_h2(const h2v w[9], const h2v a[6], Cx<float> b[6]) {
  h2v p[6], q[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    p[k] = DIR > 0 ? neg_hi(a[k]) : a[k];
    q[k] = DIR > 0 ? swp(a[k]) : neg_hi(swp(a[k]));
  }
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float re = 0.f, im = 0.f;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const h2v u = DIR > 0 ? w[i * 3 + j] : w[j * 3 + i];
        re = dot2(u, p[i * 2 + h], re);
        im = dot2(u, q[i * 2 + h], im);
      }
      b[j * 2 + h] = {re, im};
    }
}

// y = A x for one chirality: diagonal in FP32, off-diagonal entries (FP16 pairs
// cl[3..17] of the chirality) by dot2 on the FP16-rounded x
__device__ __forceinline__ void herm6_h2(const h2v* cl, const Cx<float> x[6], Cx<float> y[6]) {
  h2v X[6], Xn[6], XS[6], XSn[6];
#pragma unroll
  for (int r = 0; r < 6; ++r) {
    X[r] = to_h2(x[r]);
    Xn[r] = neg_hi(X[r]);
    XS[r] = swp(X[r]);
    XSn[r] = neg_hi(XS[r]);
  }
#pragma unroll
  for (int r = 0; r < 6; ++r) {
    const float d = (float)((r & 1) ? cl[r >> 1].y : cl[r >> 1].x);
    y[r] = cscale(d, x[r]);
  }
  int p = 3;
#pragma unroll
  for (int r = 0; r < 6; ++r)
#pragma unroll
    for (int c = r + 1; c < 6; ++c) {
      const h2v m = cl[p++];
      y[r].re = dot2(m, Xn[c], y[r].re);  // m x_c
      y[r].im = dot2(m, XS[c], y[r].im);
      y[c].re = dot2(m, X[r], y[c].re);   // conj(m) x_r
      y[c].im = dot2(m, XSn[r], y[c].im);
    }
}

__device__ __forceinline__ void clover_h2(const h2v cl[36], Cx<float> v[12]) {
  Cx<float> x[6], y0[6], y1[6];
#pragma unroll
  for (int c = 0; c < 3; ++c) { x[c] = cadd(v[c * 4 + 0], v[c * 4 + 2]); x[3 + c] = cadd(v[c * 4 + 1], v[c * 4 + 3]); }
  herm6_h2(cl, x, y0);
#pragma unroll
  for (int c = 0; c < 3; ++c) { x[c] = csub(v[c * 4 + 0], v[c * 4 + 2]); x[3 + c] = csub(v[c * 4 + 1], v[c * 4 + 3]); }
  herm6_h2(cl + 18, x, y1);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    v[c * 4 + 0] = cadd(y0[c], y1[c]);
    v[c * 4 + 2] = csub(y0[c], y1[c]);
    v[c * 4 + 1] = cadd(y0[3 + c], y1[3 + c]);
    v[c * 4 + 3] = csub(y0[3 + c], y1[3 + c]);
  }
}

}  // namespace qws
