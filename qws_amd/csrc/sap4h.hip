// sap4h.hip -- the fused SAP half-sweep on 4^4 blocks with FP16 storage: hops by link as in
// sap4.hip (a wave for the 64 links of one direction and coordinate), with the FP16
// arithmetic of sap_device.h.  The iterate, the links and the clover inverse are FP16,
// half spinors, sums and clover results FP32.
//
// The general kernel (sap_kernels.inc) reads its links from LDS at every hop, four bytes
// at a time like the iterate, 21 LDS instructions per hop.  Here the links stay in
// registers, half the size of FP32 ones, so that a wave can hold those of its own t hops as
// well, which then need no LDS; the iterate is three planes of 16 bytes.
//
// Bound by the latency of a Jacobi step (2.6 us with one workgroup on a CU) and, before
// and after, by memory.  48 KB of LDS: three workgroups per CU would fit, but 168 registers do
// not do (spills: 0.304 ms below), so two.  nm 6, the general kernel / this one: 4096 blocks
// (half of 32^3 x 64) 0.311 / 0.260 ms, 1296 blocks 0.123 / 0.102, 8 blocks 0.0287 / 0.0262;
// nm 2: 0.224 / 0.167, 0.085 / 0.062, 0.0190 / 0.0157.  (A late start of the CUs' second
// workgroups, as in sap4.hip, does not pay here: 0.260 / 0.266.)
#include "sap4_device.h"

namespace qws {

using namespace sap4;

namespace {

// Components of the iterate's LDS planes (float4 = four FP16 pairs): spins 0, 1 and 2, 3
// apart where that saves the t hops a plane.
__device__ __forceinline__ constexpr int comp(int plane, int i) {
  return plane == 0 ? (i < 2 ? i : i + 2) : plane == 1 ? 8 + i : (i < 2 ? 2 + i : 4 + i);
}
__device__ __forceinline__ void put(f4v* lx, int p, const h2v v[12]) {
  typedef _Float16 h8v __attribute__((ext_vector_type(8)));
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const h2v a = v[comp(k, 0)], b = v[comp(k, 1)], c = v[comp(k, 2)], d = v[comp(k, 3)];
    lx[k * VB + p] = __builtin_bit_cast(f4v, h8v{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y});
  }
}
// what the hop along MU, DIR takes of the spinor at LDS position p (MU < 0: all of it)
struct Raw {
  f4v q[3];
};
template <int MU, int DIR> __device__ __forceinline__ constexpr bool takes(int plane) {
  return MU != 3 || plane != (DIR > 0 ? 0 : 2);
}
template <int MU, int DIR>
__device__ __forceinline__ void read_raw(const f4v* lx, int p, Raw& r) {
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (takes<MU, DIR>(k)) r.q[k] = lx[k * VB + p];
}
template <int MU, int DIR>
__device__ __forceinline__ void unpack(const Raw& r, h2v v[12]) {
  typedef _Float16 h8v __attribute__((ext_vector_type(8)));
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const h8v h = takes<MU, DIR>(k) ? __builtin_bit_cast(h8v, r.q[k]) : h8v{};
#pragma unroll
    for (int i = 0; i < 4; ++i) v[comp(k, i)] = h2v{h[2 * i], h[2 * i + 1]};
  }
}
template <int MU, int DIR>
__device__ __forceinline__ void project_raw(const Raw& r, h2v a[6]) {
  h2v v[12];
  unpack<MU, DIR>(r, v);
  project_h2<MU, DIR>(v, a);
}

// The hops of a wave.  As in sap4.hip a wave takes the 64 links of one direction and
// coordinate, here of x, y and z only, 9 groups; a t hop ends on a lane's own site, so that
// the wave of its t slice does it and adds it up without LDS.  Three hops each, forward:
//   wave 0  x0 x1 t    wave 1  x2 y0 t    wave 2  y1 y2 t    wave 3  z0 z1 z2
// and backward:
//   wave 0  x0 x1 z2   wave 1  x2 y0 t    wave 2  y1 y2 t    wave 3  z0 z1 t
// Links: u[0], u[1] the two groups of both; u[2] z2 (waves 0, 3) or the forward t hop's;
// u[3] the backward t hop's, in wave 0 the forward one's.  ps, pn: the LDS positions of
// the ends of the first three.
struct WaveLinks {
  h2v u[4][9];
  int ps[3], pn[3];
};
template <int MU, int DIR>
__device__ __forceinline__ void task(f4v* lh, const WaveLinks& w, int i, const Raw& r) {
  h2v a[6];
  Cx<float> h[6];
  project_raw<MU, DIR>(r, a);
  link_mult_h2<DIR>(w.u[i], a, h);
  store_half(lh, MU, DIR > 0 ? w.ps[i] : w.pn[i], h);
}
template <int DIR> __device__ __forceinline__ void t_task(const h2v u[9], const Raw& r, Cx<float> acc[12]) {
  h2v a[6];
  Cx<float> h[6];
  project_raw<3, DIR>(r, a);
  link_mult_h2<DIR>(u, a, h);
  reconstruct<float, 3, DIR>(h, 2.0f, acc);
}
template <int DIR> __device__ __forceinline__ void t_task_lds(const h2v u[9], const Raw& r, f4v* t_lds, int p) {
  h2v a[6];
  Cx<float> h[6];
  project_raw<3, DIR>(r, a);
  link_mult_h2<DIR>(u, a, h);
  store_half(t_lds, 0, p, h);
}
// (T_LDS: the t hop's half spinor goes to t_lds, at p, for another wave to add)
template <int W, int DIR, bool T_LDS = false>
__device__ __forceinline__ void wave_tasks(const f4v* lx, f4v* lh, int p, const WaveLinks& w, Raw& r, Cx<float> acc[12],
                                           f4v* t_lds = nullptr) {
  constexpr int M0 = W == 3 ? 2 : W == 2 ? 1 : 0, M1 = W == 3 ? 2 : W == 0 ? 0 : 1;
  constexpr bool has_t = DIR > 0 ? W < 3 : W > 0;
  Raw r1, r2;
  read_raw<M1, DIR>(lx, DIR > 0 ? w.pn[1] : w.ps[1], r1);
  fence();
  task<M0, DIR>(lh, w, 0, r);
  fence();
  if (has_t) read_raw<3, DIR>(lx, DIR > 0 ? p + 64 : p - 64, r2);
  else read_raw<2, DIR>(lx, DIR > 0 ? w.pn[2] : w.ps[2], r2);
  fence();
  task<M1, DIR>(lh, w, 1, r1);
  fence();
  if (has_t && T_LDS) t_task_lds<DIR>(w.u[DIR > 0 && W > 0 ? 2 : 3], r2, t_lds, p);
  else if (has_t) t_task<DIR>(w.u[DIR > 0 && W > 0 ? 2 : 3], r2, acc);
  else task<2, DIR>(lh, w, 2, r2);
  fence();
}
template <int W, int DIR>
__device__ __forceinline__ void first_raw(const f4v* lx, const WaveLinks& w, Raw& r) {
  constexpr int M0 = W == 3 ? 2 : W == 2 ? 1 : 0;
  read_raw<M0, DIR>(lx, DIR > 0 ? w.pn[0] : w.ps[0], r);
}
// the x, y and z half spinors at position p into the sum, a direction at a time
template <int DIR>
__device__ __forceinline__ void sum_halves(const f4v* lh, int p, const Coord& l, Cx<float> acc[12]) {
  Halves hs;
  auto read = [&](int mu) {
#pragma unroll
    for (int k = 0; k < 3; ++k) hs.q[mu][k] = lh[(mu * 3 + k) * VB + p];
  };
  read(0), read(1);
  fence();
  if (DIR > 0 ? l.x < 3 : l.x > 0) add_half<0, DIR>(hs, 2.0f, acc);
  read(2);
  fence();
  if (DIR > 0 ? l.y < 3 : l.y > 0) add_half<1, DIR>(hs, 2.0f, acc);
  if (DIR > 0 ? l.z < 3 : l.z > 0) add_half<2, DIR>(hs, 2.0f, acc);
  fence();
}

// acc = H_in x for the iterate in lx at this thread's site (position p).
// The first barrier completes lx and frees lh; after the last one lx may be overwritten.
__device__ __forceinline__ void block_hops(const f4v* lx, f4v* lh, int wave, int p, const WaveLinks& w,
                                           Cx<float> acc[12]) {
  Raw r;
  const Coord l = coord(threadIdx.x, wave);
#pragma unroll
  for (int k = 0; k < 12; ++k) acc[k] = {0, 0};
  __syncthreads();
#define QWS_WAVE(W, DIR)              \
  first_raw<W, DIR>(lx, w, r);        \
  if (DIR < 0) __syncthreads();       \
  wave_tasks<W, DIR>(lx, lh, p, w, r, acc); \
  asm volatile("; wave %0" ::"i"(W))  /* (the branches are not merged) */
#define QWS_WAVES(DIR)                    \
  if (wave == 0) {                        \
    QWS_WAVE(0, DIR);                     \
  } else if (wave == 1) {                 \
    QWS_WAVE(1, DIR);                     \
  } else if (wave == 2) {                 \
    QWS_WAVE(2, DIR);                     \
  } else {                                \
    QWS_WAVE(3, DIR);                     \
  }
  QWS_WAVES(+1)
  __syncthreads();
  sum_halves<+1>(lh, p, l, acc);
  QWS_WAVES(-1)
  __syncthreads();
  sum_halves<-1>(lh, p, l, acc);
#undef QWS_WAVES
#undef QWS_WAVE
}

// The same with the backward hops on four more waves at the same time (helper): their half
// spinors, those of the t hops with them, in planes of their own, lb.
__device__ __forceinline__ void block_hops_wide(const f4v* lx, f4v* lh, const f4v* lb, int wave, int p, const WaveLinks& w,
                                                Cx<float> acc[12]) {
  Raw r;
  Halves hs;
  const Coord l = coord(threadIdx.x, wave);
#pragma unroll
  for (int k = 0; k < 12; ++k) acc[k] = {0, 0};
  __syncthreads();
#define QWS_WAVE(W)                                \
  first_raw<W, +1>(lx, w, r);                      \
  wave_tasks<W, +1>(lx, lh, p, w, r, acc);         \
  asm volatile("; wave %0" ::"i"(W))
  if (wave == 0) {
    QWS_WAVE(0);
  } else if (wave == 1) {
    QWS_WAVE(1);
  } else if (wave == 2) {
    QWS_WAVE(2);
  } else {
    QWS_WAVE(3);
  }
#undef QWS_WAVE
  __syncthreads();
  sum_halves<+1>(lh, p, l, acc);
#pragma unroll
  for (int k = 0; k < 3; ++k) hs.q[3][k] = lb[(9 + k) * VB + p];
  if (wave > 0) add_half<3, -1>(hs, 2.0f, acc);
  sum_halves<-1>(lb, p, l, acc);
}
__device__ __forceinline__ void helper(const f4v* lx, f4v* lb, int wave, int p, const WaveLinks& w) {
  Raw r;
  Cx<float> none[12];
  __syncthreads();
#define QWS_WAVE(W)                                             \
  first_raw<W, -1>(lx, w, r);                                   \
  wave_tasks<W, -1, true>(lx, lb, p, w, r, none, lb + 9 * VB);  \
  asm volatile("; wave %0" ::"i"(W))
  if (wave == 0) {
    QWS_WAVE(0);
  } else if (wave == 1) {
    QWS_WAVE(1);
  } else if (wave == 2) {
    QWS_WAVE(2);
  } else {
    QWS_WAVE(3);
  }
#undef QWS_WAVE
  __syncthreads();
}

// y + a x, the multiply-add written out and kept apart from a conversion to FP16 (with
// which the compiler fuses it in some places only, into one rounding), so that every
// instantiation rounds alike
__device__ __forceinline__ Cx<float> axpy(float a, Cx<float> x, Cx<float> y) {
  Cx<float> r = {fmar(a, x.re, y.re), fmar(a, x.im, y.im)};
  asm("" : "+v"(r.re), "+v"(r.im));
  return r;
}

// the block's site t of a spinor field: uniform base, 32-bit lane offset
__device__ __forceinline__ void load_site(const __half* f, long long first, long long V, unsigned t, h2v v[12]) {
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const Half4 q = (reinterpret_cast<const Half4*>(f) + (k * V + first))[t];
    v[2 * k] = __builtin_bit_cast(h2v, q.a), v[2 * k + 1] = __builtin_bit_cast(h2v, q.b);
  }
}
__device__ __forceinline__ void store_pair(__half* f, int k, long long first, long long V, unsigned t, h2v a, h2v b) {
  typedef _Float16 h4v __attribute__((ext_vector_type(4)));
  st_nt<true>(reinterpret_cast<f2v*>(f) + (k * V + first) + t, __builtin_bit_cast(f2v, h4v{a.x, a.y, b.x, b.y}));
}

// wave MU's share of the face buffer for the next launch (sap4.hip), in FP32 from the
// iterate and links as stored
template <int MU>
__device__ __forceinline__ void face_produce(const f4v* lx, int j, int p3, int p0, const Cx<float> u[9], f4v* below,
                                             f4v* above) {
  Raw r0, r1;
  h2v v[12];
  Cx<float> x[12], a[6], h[6];
  read_raw<MU, +1>(lx, p0, r0);
  read_raw<MU, -1>(lx, p3, r1);
  unpack<MU, +1>(r0, v);
#pragma unroll
  for (int k = 0; k < 12; ++k) x[k] = from_h2(v[k]);
  project<float, MU, +1>(x, a);
#pragma unroll
  for (int k = 0; k < 3; ++k)
    below[k * FS + MU * 128 + j] = f4v{a[2 * k].re, a[2 * k].im, a[2 * k + 1].re, a[2 * k + 1].im};
  unpack<MU, -1>(r1, v);
#pragma unroll
  for (int k = 0; k < 12; ++k) x[k] = from_h2(v[k]);
  project<float, MU, -1>(x, a);
  link_mult<float, -1>(u, a, h);
#pragma unroll
  for (int k = 0; k < 3; ++k)
    above[k * FS + MU * 128 + 64 + j] = f4v{h[2 * k].re, h[2 * k].im, h[2 * k + 1].re, h[2 * k + 1].im};
}

// The arguments and steps of k_sap_block_h (sap_kernels.inc), FP16 roundings in the same
// places; FB: face updates through the face buffer, else by gathers, both with the same
// roundings.  WIDE: 512 threads, waves 4 to 7 for the backward hops, as in sap4.hip; bit for
// bit the same.
template <int NL, bool FB, bool WIDE>
__global__ void __launch_bounds__(WIDE ? 2 * VB : VB, 2)
k_sap_4444_h(Geo g, const int* __restrict__ list, int nrhs, long long stride, const int* __restrict__ active, float kappa,
             int nm, int flags, __half* s, const __half* in, const __half* qface, __half* qout, __half* out,
             const __half* __restrict__ U, const __half* __restrict__ C, float* fb, long long fbs) {
  constexpr int NC = NL / 2;
  __shared__ f4v sm[(WIDE ? 24 : 12) * VB];
  f4v* lh = sm;           // half spinors, float4 [3][3][VB]; in the face update a fourth direction,
  f4v* lx = sm + 9 * VB;  // where the iterate is from then on
  f4v* lb = sm + 12 * VB;  // WIDE: the backward hops' half spinors, float4 [4][3][VB]
  const unsigned t = threadIdx.x;
  const int j = t & 63;
  const int wave8 = __builtin_amdgcn_readfirstlane(t >> 6), wave = wave8 & 3;
  const int blk = list[xcd_remap(g, blockIdx.x, gridDim.x)];
  const long long first = (long long)blk * VB, site = first + t;
  h2v cl[36];
#pragma unroll
  for (int f = 0; f < 18; ++f) {
    if (WIDE && wave8 >= 4) break;
    typedef _Float16 h4v __attribute__((ext_vector_type(4)));
    const h4v h = __builtin_bit_cast(h4v, ld_nt(reinterpret_cast<const f2v*>(C) + (f * g.V + first) + t));
    cl[2 * f] = h2v{h[0], h[1]}, cl[2 * f + 1] = h2v{h[2], h[3]};
  }
  WaveLinks wl;
  {
    Cx<float> u[4][9];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // group 2 wave + i, group 8 or a t slice
      const bool ti = i == 3 || (i == 2 && (wave == 1 || wave == 2));
      const int gi = i == 2 ? 8 : 2 * wave + i, mu = ti ? 3 : gi / 3;
      const int l = ti ? (i == 3 && wave > 0 ? wave - 1 : wave) : gi - 3 * (gi / 3);
      const unsigned ls = link_site(mu, l, j);
      if (i < 3) {
        wl.ps[i] = lds_pos(ls);
        wl.pn[i] = lds_pos(ls + (1 << (2 * mu)));
      }
#pragma unroll
      for (int k = 0; k < NC; ++k) u[i][k] = load_cx<__half>(U + 2 * (((long long)mu * NC + k) * g.V + first), ls);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (NL == 12) link_row2(u[i]);  // in FP32, then rounded
#pragma unroll
      for (int k = 0; k < 9; ++k) wl.u[i][k] = to_h2(u[i][k]);
    }
  }
  const int epi = flags & SAP_EPI_MASK;
  if (WIDE && wave8 >= 4) {  // (the barriers of the other waves' way through the loop below)
    const int p = lds_pos(t & (VB - 1));
    for (int r = blockIdx.y; r < nrhs; r += gridDim.y) {
      if (active && !active[r]) continue;
      __syncthreads();
      if (FB && (flags & SAP_FACE_PRO)) __syncthreads();
      for (int it = 0; it < nm; ++it) helper(lx, lb, wave, p, wl);
      if (epi != SAP_EPI_NONE) helper(lx, lb, wave, p, wl);
      else __syncthreads();
    }
    return;
  }
  auto face_link = [&](int j, Cx<float> u[9]) {
    const __half* Uo = opaque(U);
    const unsigned s3 = slice_site(wave, 3, j);
#pragma unroll
    for (int k = 0; k < NC; ++k) u[k] = load_cx<__half>(Uo + 2 * (((long long)wave * NC + k) * g.V + first), s3);
    if (NL == 12) link_row2(u);
  };

  int b[4], rem = blk;
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    b[m] = rem % g.NB[m];
    rem /= g.NB[m];
  }
  const float tf_hi = b[3] == g.NB[3] - 1 ? 2.0f * g.tbc : 2.0f, tf_lo = b[3] == 0 ? 2.0f * g.tbc : 2.0f;
  const int p = lds_pos(t);

  for (int r = blockIdx.y; r < nrhs; r += gridDim.y) {
    if (active && !active[r]) continue;  // uniform over the workgroup
    const long long off = r * stride;
    h2v sv[12];
    Cx<float> acc[12];
    auto hops = [&]() {
      if (WIDE) block_hops_wide(lx, lh, lb, wave, p, wl, acc);
      else block_hops(lx, lh, wave, p, wl, acc);
    };
    load_site(((flags & SAP_SRC_IN) ? in : s) + off, first, g.V, fresh_thread(), sv);
    __syncthreads();  // the previous RHS's readers of lx and lh are done
    if (flags & SAP_FACE_PRO) {
      const unsigned tt = fresh_thread();
      if constexpr (FB) {
        f4v q[6];
        Cx<float> uf[9];
        const int j = tt & 63, p3 = lds_pos(slice_site(wave, 3, j)), p0 = lds_pos(slice_site(wave, 0, j));
        read_slots(reinterpret_cast<const f4v*>(fb + r * fbs) + (long long)blk * 3 * FS, wave, j, q);
        face_link(j, uf);
        face_stage(q, wave, lh, p3, p0, uf);
        __syncthreads();
        const int pt = lds_pos(tt);
        Halves hs;  // two directions at a time
        auto read = [&](int mu) {
#pragma unroll
          for (int k = 0; k < 3; ++k) hs.q[mu][k] = lh[(mu * 3 + k) * VB + pt];
        };
        const Coord l = coord(tt, wave);
#pragma unroll
        for (int k = 0; k < 12; ++k) acc[k] = {0, 0};
        read(0), read(1);
        if (l.x == 3) add_half<0, +1>(hs, 2.0f, acc);
        if (l.x == 0) add_half<0, -1>(hs, 2.0f, acc);
        if (l.y == 3) add_half<1, +1>(hs, 2.0f, acc);
        if (l.y == 0) add_half<1, -1>(hs, 2.0f, acc);
        fence();
        read(2), read(3);
        if (l.z == 3) add_half<2, +1>(hs, 2.0f, acc);
        if (l.z == 0) add_half<2, -1>(hs, 2.0f, acc);
        if (l.t == 3) add_half<3, +1>(hs, tf_hi, acc);
        if (l.t == 0) add_half<3, -1>(hs, tf_lo, acc);
      } else {
        SiteC c;
        const long long so = opaque_v(site);
        site_coords(g, so, c);
        hop_sum<__half, NL, HOPS_FACE>(g, so, c, qface + off, opaque(U), acc);
      }
      fence();
      clover_h2(cl, acc);
#pragma unroll
      for (int k = 0; k < 12; ++k) sv[k] = to_h2(axpy(kappa, acc[k], from_h2(sv[k])));
    }

    // block solve: x_0 = s_c ; x_{k+1} = s_c + kappa T^-1 H_in x_k
    h2v x[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) x[k] = sv[k];
    put(lx, p, x);
    for (int it = 0; it < nm; ++it) {
      hops();
      fence();
      clover_h2(cl, acc);
#pragma unroll
      for (int k = 0; k < 12; ++k) x[k] = to_h2(axpy(kappa, acc[k], from_h2(sv[k])));
      put(lx, p, x);
    }
    // (a launch on the face buffer that gives s or out leaves q to nobody)
    if (!FB || epi == SAP_EPI_NONE) {
      const unsigned tq = fresh_thread();
#pragma unroll
      for (int k = 0; k < 6; ++k) store_pair(qout + off, k, first, g.V, tq, x[2 * k], x[2 * k + 1]);
    }

    if (epi != SAP_EPI_NONE) {
      // acc = T^-1 H_in x
      hops();
      const unsigned te = fresh_thread();
      h2v iv[12];
      load_site((epi == SAP_EPI_SUPDATE || (flags & SAP_SRC_IN) ? in : s) + off, first, g.V, epi == SAP_EPI_OUT ? 0 : te, iv);
      fence();
      clover_h2(cl, acc);
      // SUPDATE   s_c = s_c + in_c - x + kappa T^-1 H_in x
      // OUT       out_c = x - kappa T^-1 H_in x
      // OUT_FACE  out_c = - kappa T^-1 H_face q + x - kappa T^-1 H_in x; the face term is
      //           s_c - sv (the prologue added kappa T^-1 H_face q to s_c)
      h2v o[12];
#pragma unroll
      for (int k = 0; k < 12; ++k) {
        const Cx<float> xk = from_h2(x[k]), sk = from_h2(sv[k]), ik = from_h2(iv[k]);
        Cx<float> v;
        if (epi == SAP_EPI_SUPDATE) {
          v = axpy(kappa, acc[k], csub(cadd(sk, ik), xk));
        } else {
          v = axpy(-kappa, acc[k], xk);
          if (epi == SAP_EPI_OUT_FACE) v = cadd(v, csub(ik, sk));
        }
        o[k] = to_h2(v);
      }
      __half* dst = (epi == SAP_EPI_SUPDATE ? s : out) + off;
#pragma unroll
      for (int k = 0; k < 6; ++k) store_pair(dst, k, first, g.V, te, o[2 * k], o[2 * k + 1]);
    } else {
      __syncthreads();  // lx holds x of every site
    }
    if constexpr (FB) {
      if (flags & SAP_FACE_OUT) {
        f4v* slots = reinterpret_cast<f4v*>(fb + r * fbs);
        auto block = [&](int mu, int step) {
          const int bm = (b[mu] + step + g.NB[mu]) % g.NB[mu];
          return slots + (long long)(blk + (bm - b[mu]) * g.sN[mu]) * 3 * FS;
        };
        const int j = fresh_thread() & 63, p3 = lds_pos(slice_site(wave, 3, j)), p0 = lds_pos(slice_site(wave, 0, j));
        Cx<float> uf[9];
        face_link(j, uf);
        if (wave == 0) face_produce<0>(lx, j, p3, p0, uf, block(0, -1), block(0, +1));
        else if (wave == 1) face_produce<1>(lx, j, p3, p0, uf, block(1, -1), block(1, +1));
        else if (wave == 2) face_produce<2>(lx, j, p3, p0, uf, block(2, -1), block(2, +1));
        else face_produce<3>(lx, j, p3, p0, uf, block(3, -1), block(3, +1));
      }
    }
  }
}

}  // namespace

void launch_sap_4444_h(const Geo& g, BlockSel sel, const Batch& B, int nl, float kappa, int nm, int flags, __half* s,
                       const __half* in, const __half* qface, __half* qout, __half* out, const __half* U, const __half* C,
                       float* fb, long long fbs, hipStream_t st) {
#define SAP4H(NL, FB, WIDE)                                                                                             \
  hipLaunchKernelGGL((k_sap_4444_h<NL, FB, WIDE>), dim3(sel.n, ny), dim3(WIDE ? 2 * VB : VB), 0, st, g, sel.list, B.n, \
                     B.stride, B.active, kappa, nm, flags, s, in, qface, qout, out, U, C, fb, fbs)
#define SAP4HW(NL, FB)             \
  do {                             \
    if (wide) SAP4H(NL, FB, true); \
    else SAP4H(NL, FB, false);     \
  } while (0)
  const bool fbk = (flags & (SAP_FACE_OUT | SAP_FACE_FB)) != 0;
  const int ny = sap_rhs_groups(sel.n, B.n, 512);
  const bool wide = sel.n * ny <= WIDE_GROUPS;
  if (nl == 12) {
    if (fbk) SAP4HW(12, true);
    else SAP4HW(12, false);
  } else {
    if (fbk) SAP4HW(18, true);
    else SAP4HW(18, false);
  }
#undef SAP4HW
#undef SAP4H
}

}  // namespace qws
