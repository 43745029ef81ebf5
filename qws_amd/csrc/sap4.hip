// sap4.hip -- the fused SAP half-sweep on 4^4 blocks with FP32 storage (sap.hip has the
// method and the kernels for the other block shapes).
//
// One thread per site, as the general kernel has it, pays a full hop for the lanes that
// have no neighbour in the block (3/4 of the lanes are active), rebuilds row 2 of 12-real
// links at most hops, and leaves the waves of the two middle t slices with more work than
// the outer ones.  Here a hop is a task of its own: U a (forward) or U^+ a (backward) of
// one link inside the block, done by a wave for the 64 links of one direction and one
// coordinate l = 0..2.  4 directions x 3 coordinates = 12 link groups, three per wave:
// wave w < 3 has the x, y and z links with l = w, wave 3 the t links.  So no lane idles,
// every wave has the same work, and a thread keeps its three links (18 reals each, row 2
// rebuilt once per launch) in registers; wave mu multiplies the block faces of direction
// mu.  The half spinors go to their sites through LDS: 73.7 KB with the iterate, two
// workgroups per CU for 12-real and 18-real links alike.
//
// Bound by the latency of a Jacobi step: two waves per SIMD, four barriers, 975 vector
// instructions per wave in 7400 cycles, as long with one workgroup on the CU as with two.
// More waves do not fit: links, clover, source and sum take 251 of 256 registers.
// (Launches on few blocks have a CU for each: WIDE takes eight waves.)
// A launch on 4096 blocks (half of 32^3 x 64; nm 6), general kernel / this one: 12-real links
// 0.335 / 0.306 ms, 18-real (which the general kernel reads from memory at each hop)
// 0.564 / 0.314 ms; on 8 blocks (8^4) 0.0316 / 0.0285 ms.
#include <type_traits>

#include "kernels.h"
#include "sap.h"
#include "sap4_device.h"

namespace qws {

using namespace sap4;

namespace {

// What the hop along MU, DIR takes of the spinor at LDS position p: all six planes, or
// for t the spins 2, 3 (forward: planes 1, 3, 5) or 0, 1 (0, 2, 4).
struct Raw {
  f4v q[6];
};
template <int MU, int DIR>
__device__ __forceinline__ void read_raw(const f4v* lx, int p, Raw& r) {
#pragma unroll
  for (int k = 0; k < 6; ++k)
    if (MU < 3 || (k & 1) == (DIR > 0 ? 1 : 0)) r.q[k] = lx[k * VB + p];
}
template <int MU, int DIR>
__device__ __forceinline__ void project_raw(const Raw& r, Cx<float> a[6]) {
  Cx<float> v[12];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const bool on = MU < 3 || (k & 1) == (DIR > 0 ? 1 : 0);
    v[2 * k] = on ? Cx<float>{r.q[k].x, r.q[k].y} : Cx<float>{0, 0};
    v[2 * k + 1] = on ? Cx<float>{r.q[k].z, r.q[k].w} : Cx<float>{0, 0};
  }
  project<float, MU, DIR>(v, a);
}

// A wave's links and where their ends lie in the LDS planes.
struct WaveLinks {
  Cx<float> u[3][9];
  int ps[3], pn[3];
};

// The three tasks of a wave in direction DIR: the forward hop takes the spinor of the site
// that the link points to (position pn) and lands on the link's own site (ps), the
// backward hop the other way round.  r holds the first spinor (tasks_begin); each next
// one is read as soon as the last is projected.
template <int DIR> __device__ __forceinline__ int from(const WaveLinks& w, int i) { return DIR > 0 ? w.pn[i] : w.ps[i]; }
template <int DIR> __device__ __forceinline__ int to(const WaveLinks& w, int i) { return DIR > 0 ? w.ps[i] : w.pn[i]; }
template <int M0, int M1, int M2, int DIR>
__device__ __forceinline__ void tasks(const f4v* lx, f4v* lh, const WaveLinks& w, Raw& r) {
  Cx<float> a[6], h[6];
  project_raw<M0, DIR>(r, a);
  fence();
  read_raw<M1, DIR>(lx, from<DIR>(w, 1), r);
  fence();
  link_mult<float, DIR>(w.u[0], a, h);
  store_half(lh, M0, to<DIR>(w, 0), h);
  fence();
  project_raw<M1, DIR>(r, a);
  fence();
  read_raw<M2, DIR>(lx, from<DIR>(w, 2), r);
  fence();
  link_mult<float, DIR>(w.u[1], a, h);
  store_half(lh, M1, to<DIR>(w, 1), h);
  fence();
  project_raw<M2, DIR>(r, a);
  link_mult<float, DIR>(w.u[2], a, h);
  store_half(lh, M2, to<DIR>(w, 2), h);
}

// acc = H_in x for the iterate in lx at this thread's site (position p).
// The first barrier completes lx and frees lh; after the last one lx may be overwritten.
__device__ __forceinline__ void block_hops(const f4v* lx, f4v* lh, int wave, int p, const WaveLinks& w,
                                           Cx<float> acc[12]) {
  Raw r;
  Halves hs;
  const Coord l = coord(threadIdx.x, wave);
  __syncthreads();
  if (wave < 3) {
    read_raw<0, +1>(lx, from<+1>(w, 0), r);
    tasks<0, 1, 2, +1>(lx, lh, w, r);
    asm volatile("; x y z");  // (the two branches are not merged)
  } else {
    read_raw<3, +1>(lx, from<+1>(w, 0), r);
    tasks<3, 3, 3, +1>(lx, lh, w, r);
    asm volatile("; t");
  }
  __syncthreads();
  read_halves(lh, p, hs);
  fence();
#pragma unroll
  for (int k = 0; k < 12; ++k) acc[k] = {0, 0};
  if (l.x < 3) add_half<0, +1>(hs, 2.0f, acc);
  if (l.y < 3) add_half<1, +1>(hs, 2.0f, acc);
  if (l.z < 3) add_half<2, +1>(hs, 2.0f, acc);
  if (l.t < 3) add_half<3, +1>(hs, 2.0f, acc);
  fence();
  if (wave < 3) {
    read_raw<0, -1>(lx, from<-1>(w, 0), r);
    fence();
    __syncthreads();
    tasks<0, 1, 2, -1>(lx, lh, w, r);
    asm volatile("; x y z");
  } else {
    read_raw<3, -1>(lx, from<-1>(w, 0), r);
    fence();
    __syncthreads();
    tasks<3, 3, 3, -1>(lx, lh, w, r);
    asm volatile("; t");
  }
  __syncthreads();
  read_halves(lh, p, hs);
  fence();
  if (l.x > 0) add_half<0, -1>(hs, 2.0f, acc);
  if (l.y > 0) add_half<1, -1>(hs, 2.0f, acc);
  if (l.z > 0) add_half<2, -1>(hs, 2.0f, acc);
  if (l.t > 0) add_half<3, -1>(hs, 2.0f, acc);
}

// The same with the backward tasks on four more waves at the same time (helper), into half
// spinors of their own.
__device__ __forceinline__ void block_hops_wide(const f4v* lx, f4v* lh, int wave, int p, const WaveLinks& w,
                                                Cx<float> acc[12]) {
  Raw r;
  Halves hs;
  const Coord l = coord(threadIdx.x, wave);
  __syncthreads();
  if (wave < 3) {
    read_raw<0, +1>(lx, from<+1>(w, 0), r);
    tasks<0, 1, 2, +1>(lx, lh, w, r);
    asm volatile("; x y z");
  } else {
    read_raw<3, +1>(lx, from<+1>(w, 0), r);
    tasks<3, 3, 3, +1>(lx, lh, w, r);
    asm volatile("; t");
  }
  __syncthreads();
  read_halves(lh, p, hs);
  fence();
#pragma unroll
  for (int k = 0; k < 12; ++k) acc[k] = {0, 0};
  if (l.x < 3) add_half<0, +1>(hs, 2.0f, acc);
  if (l.y < 3) add_half<1, +1>(hs, 2.0f, acc);
  if (l.z < 3) add_half<2, +1>(hs, 2.0f, acc);
  if (l.t < 3) add_half<3, +1>(hs, 2.0f, acc);
  fence();
  read_halves(lh + 12 * VB, p, hs);
  fence();
  if (l.x > 0) add_half<0, -1>(hs, 2.0f, acc);
  if (l.y > 0) add_half<1, -1>(hs, 2.0f, acc);
  if (l.z > 0) add_half<2, -1>(hs, 2.0f, acc);
  if (l.t > 0) add_half<3, -1>(hs, 2.0f, acc);
}
__device__ __forceinline__ void helper(const f4v* lx, f4v* lh, int wave, const WaveLinks& w) {
  Raw r;
  __syncthreads();
  if (wave < 3) {
    read_raw<0, -1>(lx, from<-1>(w, 0), r);
    tasks<0, 1, 2, -1>(lx, lh + 12 * VB, w, r);
    asm volatile("; x y z");
  } else {
    read_raw<3, -1>(lx, from<-1>(w, 0), r);
    tasks<3, 3, 3, -1>(lx, lh + 12 * VB, w, r);
    asm volatile("; t");
  }
  __syncthreads();
}

// The block's site t of a spinor field: uniform base, 32-bit lane offset (no 64-bit
// address per plane in vector registers).
__device__ __forceinline__ void load_site(const float* f, long long first, long long V, unsigned t, Cx<float> v[12]) {
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const f4v q = (reinterpret_cast<const f4v*>(f) + (k * V + first))[t];
    v[2 * k] = {q.x, q.y};
    v[2 * k + 1] = {q.z, q.w};
  }
}

// Wave MU's share of the face buffer for the next launch: this block's l = 0 sites as
// the + side of the block below, its l = 3 sites through their links as the - side of
// the block above.
template <int MU>
__device__ __forceinline__ void face_produce(const f4v* lx, int j, int p3, int p0, const Cx<float> u[9],
                                             f4v* below, f4v* above) {
  Raw r0, r1;
  Cx<float> a[6], h[6];
  read_raw<MU, +1>(lx, p0, r0);
  read_raw<MU, -1>(lx, p3, r1);
  project_raw<MU, +1>(r0, a);
#pragma unroll
  for (int k = 0; k < 3; ++k)
    below[k * FS + MU * 128 + j] = f4v{a[2 * k].re, a[2 * k].im, a[2 * k + 1].re, a[2 * k + 1].im};
  project_raw<MU, -1>(r1, a);
  link_mult<float, -1>(u, a, h);
#pragma unroll
  for (int k = 0; k < 3; ++k)
    above[k * FS + MU * 128 + 64 + j] = f4v{h[2 * k].re, h[2 * k].im, h[2 * k + 1].re, h[2 * k + 1].im};
}

// The arguments and steps of k_sap_block (sap_kernels.inc); FB: face updates through the
// face buffer, else by gathers, both with the same roundings.  WIDE: 512 threads, waves 4
// to 7 for the backward tasks, one workgroup per CU (123 KB of LDS); bit for bit the same.
template <int NL, bool FB, bool MULTI, bool WIDE>
__global__ void __launch_bounds__(WIDE ? 2 * VB : VB, 2)
k_sap_4444(Geo g, const int* __restrict__ list, int nrhs, long long stride, const int* __restrict__ active, float kappa,
           int nm, int flags, float* s, const float* in, const float* qface, float* qout, float* out,
           const float* __restrict__ U, const float* __restrict__ C, float* fb, long long fbs, SapSrcUpdate upd,
           SapMulti<float> multi) {
  constexpr int NC = NL / 2;
  __shared__ f4v sm[(6 + (WIDE ? 24 : 12)) * VB];
  f4v* lx = sm;           // the iterate, float4 [6][VB]
  f4v* lh = sm + 6 * VB;  // half spinors, float4 [4][3][VB] (WIDE: of each direction)
  const unsigned t = threadIdx.x;
  const int j = t & 63;
  const int wave8 = __builtin_amdgcn_readfirstlane(t >> 6), wave = wave8 & 3;
  int blk;
  if constexpr (MULTI) {
    const int2 e = multi.table[xcd_remap_n(multi.xcd, blockIdx.x, gridDim.x)];
    const SapPart<float>& P = multi.parts[e.x];
    g = P.g, active = P.active, stride = P.stride, nrhs = P.nrhs, kappa = P.kappa;
    s = P.s, in = P.in, qface = P.qface, qout = P.qout, out = P.out, U = P.U, C = P.C, fb = P.fb, fbs = P.fbs;
    upd = P.upd;
    blk = e.y;
  } else {
    blk = list[xcd_remap(g, blockIdx.x, gridDim.x)];
  }
  // The two workgroups of a CU would load, solve and write at the same time: in a launch
  // of several rounds the second ones start half a block's time late (a sleep of about
  // 1 us each turn), so that one computes while the other waits for memory.  SAP launch,
  // without and with it (nm 6): 4096 blocks 0.316 / 0.308 ms, 2048 blocks 0.170 / 0.162;
  // 512 blocks, a single round, 0.049 / 0.055, so not there.
  if (gridDim.x >= 1024 && blockIdx.y == 0 && blockIdx.x >= 256 && blockIdx.x < 512)
    for (int i = 6 + nm * 8 / 5; i > 0; --i) __builtin_amdgcn_s_sleep(37);
  const long long first = (long long)blk * VB, site = first + t;
  CloverRegs<float> cl;
  if (!WIDE || wave8 < 4) cl.load(C, site, g.V);

  WaveLinks wl;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int mu = wave < 3 ? i : 3;
    const unsigned ls = link_site(mu, wave < 3 ? wave : i, j);
    wl.ps[i] = lds_pos(ls);
    wl.pn[i] = lds_pos(ls + (1 << (2 * mu)));
#pragma unroll
    for (int k = 0; k < NC; ++k) wl.u[i][k] = load_cx<float>(U + 2 * (((long long)mu * NC + k) * g.V + first), ls);
  }
  const int epi = flags & SAP_EPI_MASK;
  if (WIDE && wave8 >= 4) {  // (the barriers of the other waves' way through the loop below)
    if (NL == 12) {
#pragma unroll
      for (int i = 0; i < 3; ++i) link_row2(wl.u[i]);
    }
    for (int r = blockIdx.y; r < nrhs; r += gridDim.y) {
      if (active && !active[r]) continue;
      __syncthreads();
      if (FB && (flags & SAP_FACE_PRO)) __syncthreads();
      for (int it = 0; it < nm; ++it) helper(lx, lh, wave, wl);
      if (epi != SAP_EPI_NONE) helper(lx, lh, wave, wl);
      else __syncthreads();
    }
    return;
  }
  // the wave's face links, loaded where they are used (they are in cache, and there are
  // no registers to keep them in during the block solve)
  auto face_link = [&](int j, Cx<float> u[9]) {
    const float* Uo = opaque(U);
    const unsigned s3 = slice_site(wave, 3, j);
#pragma unroll
    for (int k = 0; k < NC; ++k) u[k] = load_cx<float>(Uo + 2 * (((long long)wave * NC + k) * g.V + first), s3);
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
    Cx<float> sv[12], acc[12];
    auto hops = [&]() {
      if (WIDE) block_hops_wide(lx, lh, wave, p, wl, acc);
      else block_hops(lx, lh, wave, p, wl, acc);
    };
    if (flags & SAP_SRC_PUPD) src_update(upd, r, off, opaque_v(site), g.V);
    // every load of the prologue is issued here, with those of the links and the clover
    // still on their way (one round trip to memory, not three)
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
        fence();
        if (NL == 12) link_row2(uf);
        face_stage(q, wave, lh, p3, p0, uf);
        __syncthreads();
        Halves hs;
        read_halves(lh, lds_pos(tt), hs);
        fence();
        const Coord l = coord(tt, wave);
#pragma unroll
        for (int k = 0; k < 12; ++k) acc[k] = {0, 0};
        if (l.x == 3) add_half<0, +1>(hs, 2.0f, acc);
        if (l.x == 0) add_half<0, -1>(hs, 2.0f, acc);
        if (l.y == 3) add_half<1, +1>(hs, 2.0f, acc);
        if (l.y == 0) add_half<1, -1>(hs, 2.0f, acc);
        if (l.z == 3) add_half<2, +1>(hs, 2.0f, acc);
        if (l.z == 0) add_half<2, -1>(hs, 2.0f, acc);
        if (l.t == 3) add_half<3, +1>(hs, tf_hi, acc);
        if (l.t == 0) add_half<3, -1>(hs, tf_lo, acc);
      } else {
        SiteC c;
        const long long so = opaque_v(site);
        site_coords(g, so, c);
        hop_sum<float, NL, HOPS_FACE>(g, so, c, qface + off, opaque(U), acc);
      }
      fence();
      clover_regs(cl, acc);
      fence();
#pragma unroll
      for (int k = 0; k < 12; ++k) sv[k] = {sv[k].re + kappa * acc[k].re, sv[k].im + kappa * acc[k].im};
    }

    // block solve: x_0 = s_c ; x_{k+1} = s_c + kappa T^-1 H_in x_k
    auto put = [&](const Cx<float> v[12]) {
#pragma unroll
      for (int k = 0; k < 6; ++k)
        lx[k * VB + p] = f4v{v[2 * k].re, v[2 * k].im, v[2 * k + 1].re, v[2 * k + 1].im};
    };
    put(sv);
    if (NL == 12) {  // (again for each RHS: there are no registers for it during the face update)
#pragma unroll
      for (int i = 0; i < 3; ++i) link_row2(wl.u[i]);
    }
    fence();
    for (int it = 0; it < nm; ++it) {
      hops();
      fence();
      clover_regs(cl, acc);
#pragma unroll
      for (int k = 0; k < 12; ++k) acc[k] = cadd(sv[k], cscale(kappa, acc[k]));
      put(acc);
    }
    // (a launch on the face buffer that gives s or out leaves q to nobody)
    if (!FB || epi == SAP_EPI_NONE) {
      const unsigned tq = fresh_thread();
#pragma unroll
      for (int k = 0; k < 6; ++k) (reinterpret_cast<f4v*>(qout + off) + (k * g.V + first))[tq] = lx[k * VB + p];
    }

    if (epi != SAP_EPI_NONE) {
      // acc = T^-1 H_in x
      hops();
      const unsigned te = fresh_thread();
      // (SAP_EPI_OUT takes nothing: one line of s for all threads, so that the loads need no branch)
      const float* src = epi == SAP_EPI_SUPDATE || (flags & SAP_SRC_IN) ? in : s;
      const unsigned ti = epi == SAP_EPI_OUT ? 0 : te;
      const f4v* pi = reinterpret_cast<const f4v*>(src + off) + first;
      f4v iv[6];
#pragma unroll
      for (int k = 0; k < 6; ++k) iv[k] = (pi + k * g.V)[ti];
      fence();
      clover_regs(cl, acc);
      fence();
      // a plane at a time: x again (kept in LDS, not in registers, meanwhile) and
      //   SUPDATE   s_c = s_c + in_c - x + kappa T^-1 H_in x
      //   OUT       out_c = x - kappa T^-1 H_in x
      //   OUT_FACE  out_c = - kappa T^-1 H_face q + x - kappa T^-1 H_in x; the face term is
      //             s_c - sv (the prologue added kappa T^-1 H_face q to s_c)
      float* dst = epi == SAP_EPI_SUPDATE ? s : out;
      f4v* po = reinterpret_cast<f4v*>(dst + off) + first;
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        const f4v xk = lx[k * VB + p];
        const f4v ak = {acc[2 * k].re, acc[2 * k].im, acc[2 * k + 1].re, acc[2 * k + 1].im};
        const f4v sk = {sv[2 * k].re, sv[2 * k].im, sv[2 * k + 1].re, sv[2 * k + 1].im};
        f4v o;
        if (epi == SAP_EPI_SUPDATE) {
          o = ((sk + iv[k]) - xk) + kappa * ak;
        } else {
          o = xk - kappa * ak;
          if (epi == SAP_EPI_OUT_FACE) o = o + (iv[k] - sk);
        }
        st_nt<true>((po + k * g.V) + te, o);
        fence();
      }
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
        if (NL == 12) link_row2(uf);
        if (wave == 0) face_produce<0>(lx, j, p3, p0, uf, block(0, -1), block(0, +1));
        else if (wave == 1) face_produce<1>(lx, j, p3, p0, uf, block(1, -1), block(1, +1));
        else if (wave == 2) face_produce<2>(lx, j, p3, p0, uf, block(2, -1), block(2, +1));
        else face_produce<3>(lx, j, p3, p0, uf, block(3, -1), block(3, +1));
      }
    }
  }
}

}  // namespace

bool sap_is_4444(const Geo& g) { return g.B[0] == 4 && g.B[1] == 4 && g.B[2] == 4 && g.B[3] == 4; }

void launch_sap_4444(const Geo& g, BlockSel sel, const Batch& B, int nl, float kappa, int nm, int flags, float* s,
                     const float* in, const float* qface, float* qout, float* out, const float* U, const float* C,
                     float* fb, long long fbs, hipStream_t st, const SapSrcUpdate& upd) {
#define SAP4(NL, FB, WIDE)                                                                                              \
  hipLaunchKernelGGL((k_sap_4444<NL, FB, false, WIDE>), dim3(sel.n, ny), dim3(WIDE ? 2 * VB : VB), 0, st, g, sel.list, B.n, B.stride, B.active, \
                     kappa, nm, flags, s, in, qface, qout, out, U, C, fb, fbs, upd, SapMulti<float>())
  const bool fbk = (flags & (SAP_FACE_OUT | SAP_FACE_FB)) != 0;
  const int ny = sap_rhs_groups(sel.n, B.n, 512);
  const bool wide = sel.n * ny <= WIDE_GROUPS;
#define SAP4W(NL, FB)             \
  do {                            \
    if (wide) SAP4(NL, FB, true); \
    else SAP4(NL, FB, false);     \
  } while (0)
  if (nl == 12) {
    if (fbk) SAP4W(12, true);
    else SAP4W(12, false);
  } else {
    if (fbk) SAP4W(18, true);
    else SAP4W(18, false);
  }
#undef SAP4W
#undef SAP4
}

void launch_sap_4444_multi(const SapMulti<float>& m, int nl, int nm, int flags, hipStream_t st) {
  const Geo g0{};
  const SapSrcUpdate u0;
#define SAP4(NL, FB, WIDE)                                                                                               \
  hipLaunchKernelGGL((k_sap_4444<NL, FB, true, WIDE>), dim3(m.n, m.rhs), dim3(WIDE ? 2 * VB : VB), 0, st, g0, nullptr, 0, 0, nullptr, 0.0f, nm, flags, \
                     nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, u0, m)
  const bool fbk = (flags & (SAP_FACE_OUT | SAP_FACE_FB)) != 0;
  const bool wide = m.n * m.rhs <= WIDE_GROUPS;
#define SAP4W(NL, FB)             \
  do {                            \
    if (wide) SAP4(NL, FB, true); \
    else SAP4(NL, FB, false);     \
  } while (0)
  if (nl == 12) {
    if (fbk) SAP4W(12, true);
    else SAP4W(12, false);
  } else {
    if (fbk) SAP4W(18, true);
    else SAP4W(18, false);
  }
#undef SAP4W
#undef SAP4
}

}  // namespace qws
