// eo.hip -- the even/odd operator family (deo_*, dee_deo_*, one_minus_*, mtilde) on
// x-compressed parity fields.
//
// A parity-p field holds Vh = V/2 sites h = xh + (Lx/2)(y + Ly(z + Lz t)); its row
// parity is ick = (p + y + z + t) % 2 (deo_in_d.cc:80-85).  Neighbours follow the
// reference's index arithmetic: x-forward of h is xh (ick 0) or xh + 1 (ick 1) of
// the other parity, x-backward xh - 1 (ick 0) or xh (ick 1); y/z/t keep xh; every
// index wraps.  With even extents this is the physical lattice with x = 2 xh + ick.
// Device layout per parity (site-major SoA like the blocked layout):
//   spinor  FP32 float4 [6][Vh], FP64 double2 [12][Vh]
//   links   [2][4][NL/2][Vh] Vec2  (link from site h of parity p)
//   clover  [2][18][Vh] float4 / [2][36][Vh] double2
// One thread per site of the output parity, or four on few sites.
#include <stdexcept>
#include <type_traits>

#include "kernels.h"
#include "split_device.h"

namespace qws {

constexpr int EO_THREADS = 256;

// Whether k_deo reads links and clover and writes its output past the caches (NT): it uses
// each link and clover once, so that they only push out the spinors, which it reads eight
// times.  Where the operator's data fit the last-level cache, its next application takes
// them from there.  mtilde, us with ordinary / nontemporal accesses, by MB per k_deo:
//   FP32 138 43.4 / 50.8   191 76.5 / 83.1   207 80.0 / 75.6   233 93.2 / 93.8   350 157 / 145   906 397 / 332
//   FP64  69 30.2 / 39.8   138 52.6 / 50.0   207 86.7 / 85.0   277  117 / 99.5   701 330 / 276  2214 1031 / 830
constexpr double DEO_STREAM_BYTES = 200e6;

struct EoSite {
  int c[4];  // xh, y, z, t
  int ick;
};

// What the operator takes of Geo: a launch copies its arguments, and the kernel's first
// loads fetch them from the host (mtilde FP32 12-real with all of Geo / so: 8^4 9.74 / 8.82 us,
// 16^3 48 32.3 / 31.4).
struct EoGeo {
  int L[4];
  int tbc, xcd_remap;
  long long V;
};

template <typename G> __device__ __forceinline__ void eo_coords(const G& g, int pe, long long h, EoSite& e) {
  const int nxh = g.L[0] >> 1;
  long long r = h;
  e.c[0] = (int)(r % nxh); r /= nxh;
  e.c[1] = (int)(r % g.L[1]); r /= g.L[1];
  e.c[2] = (int)(r % g.L[2]);
  e.c[3] = (int)(r / g.L[2]);
  e.ick = (pe + e.c[1] + e.c[2] + e.c[3]) & 1;
}

// One hop of H (or of H^+: projector and reconstruction of the opposite direction,
// deo_dag_in.cc) into acc; set 1 skips hops that wrap round the lattice ("_in_"),
// set 2 keeps only those ("_out_pre/_pos"), whose t edge carries 2*tbc.
template <typename S, int NL, int MU, int DIR, bool DAG, bool NT>
__device__ __forceinline__ void eo_hop(const EoGeo& g, int pe, long long h, const EoSite& e, int set, const S* in,
                                       const S* U, long long Vh, Cx<typename Store<S>::R> acc[12]) {
  using R = typename Store<S>::R;
  const int nxh = g.L[0] >> 1;
  int n[4] = {e.c[0], e.c[1], e.c[2], e.c[3]};
  bool wraps;
  if (MU == 0) {
    const int v = e.c[0] + (DIR > 0 ? e.ick : e.ick - 1);
    wraps = v < 0 || v >= nxh;
    n[0] = v < 0 ? nxh - 1 : (v >= nxh ? 0 : v);
  } else {
    const int ext = g.L[MU];
    const int v = e.c[MU] + DIR;
    wraps = v < 0 || v >= ext;
    n[MU] = v < 0 ? ext - 1 : (v >= ext ? 0 : v);
  }
  if ((set == 1 && wraps) || (set == 2 && !wraps)) return;
  const long long hn = n[0] + (long long)nxh * (n[1] + (long long)g.L[1] * (n[2] + (long long)g.L[2] * n[3]));
  constexpr int PD = DAG ? -DIR : DIR;
  Cx<R> v[12], a[6], b[6], u[9];
  SpinorIO<S>::load(in, hn, Vh, v);
  project<R, MU, PD>(v, a);
  // forward: the link of h (parity pe); backward: the link of the neighbour (parity 1-pe)
  const S* Ub = U + (long long)(DIR > 0 ? pe : 1 - pe) * 4 * NL * Vh;
  load_link<S, NL, NT>(Ub, MU, DIR > 0 ? h : hn, Vh, u);
  link_mult<R, DIR>(u, a, b);
  const R tf = (MU == 3 && wraps) ? (R)(2 * g.tbc) : (R)2;
  reconstruct<R, MU, PD>(b, tf, acc);
}

// Reductions of out that BiCGStab takes next, in FP64 without another pass over it:
// <z, out> (DEO_DOT) or |out|^2 and <out, in0> (DEO_NORM_DOT).
template <int RED, typename R>
__device__ __forceinline__ void deo_reduce(Cx<R> o, Cx<R> w, double acc[3]) {
  if (RED == DEO_DOT) {
    acc[0] += (double)w.re * o.re + (double)w.im * o.im;
    acc[1] += (double)w.re * o.im - (double)w.im * o.re;
  } else if (RED == DEO_NORM_DOT) {
    acc[0] += (double)o.re * o.re + (double)o.im * o.im;
    acc[1] += (double)o.re * w.re + (double)o.im * w.im;
    acc[2] += (double)o.re * w.im - (double)o.im * w.re;
  }
}
// the workgroup's sums: part[v * gridDim.x + blockIdx.x]
template <int RED> __device__ __forceinline__ void deo_partials(const double acc[3], double* part) {
  __shared__ double sh[3][EO_THREADS / 64];
  constexpr int NV = RED == DEO_DOT ? 2 : 3;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    double x = acc[v];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
    if ((threadIdx.x & 63) == 0) sh[v][threadIdx.x >> 6] = x;
  }
  __syncthreads();
  if (threadIdx.x < NV)
    part[(long long)threadIdx.x * gridDim.x + blockIdx.x] =
        ((sh[threadIdx.x][0] + sh[threadIdx.x][1]) + sh[threadIdx.x][2]) + sh[threadIdx.x][3];
}

// For every site h of parity pe: acc = sum of the hops of `set` (0 all, 1 no wrap,
// 2 wrap only, 3 none: acc = in[h]) from in; clv: acc = T^-1 acc; then
// mode 0: out = acc, 1: out += fac acc, 2: out = in0 + fac acc.
template <typename S, int NL, bool DAG, bool NT, int RED>
__global__ void __launch_bounds__(EO_THREADS)
k_deo(EoGeo g, int pe, int set, int clv, int mode, typename Store<S>::R fac, S* out, const S* __restrict__ in,
      const S* in0, const S* __restrict__ U, const S* __restrict__ C, const S* z, double* part) {
  using R = typename Store<S>::R;
  const long long Vh = g.V >> 1;
  // XCD-contiguous ranges of sites: the z and t neighbours a workgroup reads were fetched
  // by workgroups on the same XCD (its L2), not by ones spread round-robin over the XCDs
  long long h = xcd_remap_n(g.xcd_remap, blockIdx.x, gridDim.x) * (long long)EO_THREADS + threadIdx.x;
  const bool on = h < Vh;
  if (RED == DEO_STORE && !on) return;
  if (!on) h = Vh - 1;  // (idle, but there for the sums)
  EoSite e;
  eo_coords(g, pe, h, e);
  Cx<R> acc[12];
  if (set == 3) {
    SpinorIO<S>::load(in, h, Vh, acc);
  } else {
#pragma unroll
    for (int k = 0; k < 12; ++k) acc[k] = {0, 0};
    eo_hop<S, NL, 0, +1, DAG, NT>(g, pe, h, e, set, in, U, Vh, acc);
    eo_hop<S, NL, 0, -1, DAG, NT>(g, pe, h, e, set, in, U, Vh, acc);
    eo_hop<S, NL, 1, +1, DAG, NT>(g, pe, h, e, set, in, U, Vh, acc);
    eo_hop<S, NL, 1, -1, DAG, NT>(g, pe, h, e, set, in, U, Vh, acc);
    eo_hop<S, NL, 2, +1, DAG, NT>(g, pe, h, e, set, in, U, Vh, acc);
    eo_hop<S, NL, 2, -1, DAG, NT>(g, pe, h, e, set, in, U, Vh, acc);
    eo_hop<S, NL, 3, +1, DAG, NT>(g, pe, h, e, set, in, U, Vh, acc);
    eo_hop<S, NL, 3, -1, DAG, NT>(g, pe, h, e, set, in, U, Vh, acc);
  }
  if (clv) clover_apply<S, NT>(C + (long long)pe * 72 * Vh, h, Vh, acc);
  double red[3] = {0, 0, 0};
  if (mode != 0) {
    Cx<R> o[12];
    SpinorIO<S>::load(mode == 1 ? out : in0, h, Vh, o);
#pragma unroll
    for (int k = 0; k < 12; ++k) acc[k] = cadd(o[k], cscale(fac, acc[k]));
    if (RED == DEO_DOT) SpinorIO<S>::load(z, h, Vh, o);
    if (RED != DEO_STORE && on) {
#pragma unroll
      for (int k = 0; k < 12; ++k) deo_reduce<RED>(acc[k], o[k], red);
    }
  }
  if (RED == DEO_STORE || on) SpinorIO<S>::template store<NT>(out, h, Vh, acc);
  if (RED != DEO_STORE) deo_partials<RED>(red, part);
}

// k_deo (sets 0 to 2) with four waves per 64 sites, for few sites: as k_split of split.hip.
template <typename S, int NL, int MU, bool DAG, typename Rest>
__device__ __forceinline__ void eo_two_hops(const EoGeo& g, int pe, int h, int first, const EoSite& e, bool on, int set,
                                            const S* in, const S* U, Cx<typename Store<S>::R> (*lh)[6][split::SITES],
                                            Rest&& rest) {
  using R = typename Store<S>::R;
  using IO = split::IO<S>;
  constexpr int NC = NL / 2, BOTH = sizeof(S) == 8 ? 0 : 1;
  const int lane = threadIdx.x & 63, Vh = (int)(g.V >> 1), nxh = g.L[0] >> 1;
  const int step = MU == 0 ? 1 : MU == 1 ? nxh : MU == 2 ? nxh * g.L[1] : nxh * g.L[1] * g.L[2];
  Cx<R> v[1 + BOTH][12], u[1 + BOTH][9];
  bool take[2];
  auto load = [&](int d) {
    const int ext = MU == 0 ? nxh : g.L[MU], dir = d == 0 ? 1 : -1;
    const int c = e.c[MU] + (MU == 0 ? (d == 0 ? e.ick : e.ick - 1) : dir);
    const bool wraps = c < 0 || c >= ext;
    const int n = h + ((c < 0 ? ext - 1 : c >= ext ? 0 : c) - e.c[MU]) * step;
    take[d] = on && !((set == 1 && wraps) || (set == 2 && !wraps));
    if (!__any(take[d])) return;
    const unsigned nn = take[d] ? n : first, at = d == 0 ? (take[d] ? h : first) : nn;
    const S* Ub = U + (long long)(d == 0 ? pe : 1 - pe) * 4 * NL * Vh;
#pragma unroll
    for (int j = 0; j < 6; ++j) IO::load2(in, j, Vh, nn * IO::Q, v[d * BOTH] + 2 * j);
#pragma unroll
    for (int k = 0; k < NC; ++k) u[d * BOTH][k] = IO::link(Ub, MU * NC + k, Vh, at * split::LINK_BYTES<S>);
  };
  auto hop = [&](int d) {
    Cx<R> o[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) o[k] = {0, 0};
    if (__any(take[d])) {
      Cx<R> a[6], m[6];
      if (NL == 12) link_row2(u[d * BOTH]);
      if (d == 0) {
        project<R, MU, DAG ? -1 : +1>(v[d * BOTH], a);
        link_mult<R, +1>(u[d * BOTH], a, m);
      } else {
        project<R, MU, DAG ? +1 : -1>(v[d * BOTH], a);
        link_mult<R, -1>(u[d * BOTH], a, m);
      }
#pragma unroll
      for (int k = 0; k < 6; ++k) o[k] = {take[d] ? m[k].re : R(0), take[d] ? m[k].im : R(0)};
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) lh[2 * MU + d][k][lane] = o[k];
  };
  asm volatile("; hops of direction %0" ::"i"(MU));  // (the four waves' branches are not merged)
  load(0);
  if (BOTH) load(1);
  if (BOTH) rest();
  __builtin_amdgcn_sched_barrier(0);
  hop(0);
  if (!BOTH) {
    load(1);
    hop(1);
    rest();
  } else {
    hop(1);
  }
  asm volatile("; end of direction %0" ::"i"(MU));
}

template <typename S, int NL, bool DAG, int RED>
__global__ void __launch_bounds__(256, 2)
k_deo_split(EoGeo g, float rnx, float ry, float rz, int pe, int set, int clv, int mode, typename Store<S>::R fac, S* out,
            const S* __restrict__ in, const S* in0, const S* __restrict__ U, const S* __restrict__ C, const S* z,
            double* part) {
  using R = typename Store<S>::R;
  using IO = split::IO<S>;
  constexpr int SITES = split::SITES;
  __shared__ Cx<R> lh[8][6][SITES];
  __shared__ Cx<R> ly[12][SITES];
  const int lane = threadIdx.x & 63, Vh = (int)(g.V >> 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int first = xcd_remap_n(g.xcd_remap, blockIdx.x, gridDim.x) * SITES;
  const bool on = first + lane < Vh;
  const int h = on ? first + lane : first;
  EoSite e;
  {
    // quotients by the reciprocal: exact below 2^20
    const int nxh = g.L[0] >> 1;
    const int q0 = (int)((h + 0.5f) * rnx), q1 = (int)((q0 + 0.5f) * ry), q2 = (int)((q1 + 0.5f) * rz);
    e.c[0] = h - q0 * nxh, e.c[1] = q0 - q1 * g.L[1], e.c[2] = q1 - q2 * g.L[2], e.c[3] = q2;
    e.ick = (pe + e.c[1] + e.c[2] + e.c[3]) & 1;
  }
  const unsigned at = (unsigned)h * IO::Q;
  R ca[36];  // chirality wave & 1 of T^-1
  auto rest = [&]() { IO::chir(C + (long long)pe * 72 * Vh, wave & 1, Vh, at, ca); };  // (unused without clv)
  if (wave == 0) eo_two_hops<S, NL, 0, DAG>(g, pe, h, first, e, on, set, in, U, lh, rest);
  else if (wave == 1) eo_two_hops<S, NL, 1, DAG>(g, pe, h, first, e, on, set, in, U, lh, rest);
  else if (wave == 2) eo_two_hops<S, NL, 2, DAG>(g, pe, h, first, e, on, set, in, U, lh, rest);
  else eo_two_hops<S, NL, 3, DAG>(g, pe, h, first, e, on, set, in, U, lh, rest);
  __syncthreads();
  Cx<R> acc[12], b[6];
#pragma unroll
  for (int k = 0; k < 12; ++k) acc[k] = {0, 0};
  const R tf_hi = e.c[3] == g.L[3] - 1 ? (R)(2 * g.tbc) : R(2), tf_lo = e.c[3] == 0 ? (R)(2 * g.tbc) : R(2);
#define ADD(MU, DIR, TF)                                                                       \
  _Pragma("unroll") for (int k = 0; k < 6; ++k) b[k] = lh[2 * MU + (DIR < 0)][k][lane];        \
  reconstruct<R, MU, DAG ? -(DIR) : DIR>(b, TF, acc);
  ADD(0, +1, R(2)) ADD(0, -1, R(2)) ADD(1, +1, R(2)) ADD(1, -1, R(2))
  ADD(2, +1, R(2)) ADD(2, -1, R(2)) ADD(3, +1, tf_hi) ADD(3, -1, tf_lo)
#undef ADD
  // wave c < 3 stores colour c; its term of the output, and of the sums
  Cx<R> o[2][2], w[2][2];
  auto terms = [&]() {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (mode != 0) IO::load2(mode == 1 ? out : in0, 2 * wave + j, Vh, at, o[j]);
      if (RED == DEO_DOT) IO::load2(z, 2 * wave + j, Vh, at, w[j]);
    }
  };
  if (sizeof(S) == 4 && wave < 3) terms();  // (FP64 has no registers for them yet)
  if (clv) {
    Cx<R> x[6], y[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if (wave & 1) x[c] = csub(acc[c * 4], acc[c * 4 + 2]), x[3 + c] = csub(acc[c * 4 + 1], acc[c * 4 + 3]);
      else x[c] = cadd(acc[c * 4], acc[c * 4 + 2]), x[3 + c] = cadd(acc[c * 4 + 1], acc[c * 4 + 3]);
    }
    if (wave < 2) split::herm3_mult<0>(ca, x, y);
    else split::herm3_mult<1>(ca, x, y);
#pragma unroll
    for (int k = 0; k < 3; ++k) ly[(wave & 1) * 6 + (wave >> 1) * 3 + k][lane] = y[k];
  } else if (wave == 0) {  // as the two chiralities whose combination is acc
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      ly[c][lane] = acc[4 * c], ly[3 + c][lane] = acc[4 * c + 1];
      ly[6 + c][lane] = acc[4 * c + 2], ly[9 + c][lane] = acc[4 * c + 3];
    }
  }
  __syncthreads();
  double red[3] = {0, 0, 0};
  if (wave < 3 && on) {
    if (sizeof(S) == 8) terms();
    const Cx<R> y0 = ly[wave][lane], y1 = ly[3 + wave][lane], z0 = ly[6 + wave][lane], z1 = ly[9 + wave][lane];
    Cx<R> t[2][2] = {{y0, y1}, {z0, z1}};
    if (clv) t[0][0] = cadd(y0, z0), t[0][1] = cadd(y1, z1), t[1][0] = csub(y0, z0), t[1][1] = csub(y1, z1);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (mode != 0) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          t[j][k] = cadd(o[j][k], cscale(fac, t[j][k]));
          if (RED != DEO_STORE) deo_reduce<RED>(t[j][k], RED == DEO_DOT ? w[j][k] : o[j][k], red);
        }
      }
      IO::store2(out, 2 * wave + j, Vh, at, t[j]);
    }
  }
  if (RED != DEO_STORE) deo_partials<RED>(red, part);
}

// Whether k_deo_split is the faster one: by its workgroups (64 sites), where it is no slower
// with three lattices on a stream each in turn / with one again and again.  mtilde in us, k_deo,
// then it:
//   workgroups      32                 256               1024                1280
//   FP32 12-real    7.9/16.6 7.8/8.8   8.6/17.1 7.9/9.3  18.2/26.1 17.1/24.0 22.6/29.6 21.1/27.7
//        18-real    7.7/16.5 6.3/10.0  9.2/17.8 6.3/10.4 20.8/28.1 20.3/27.3 27.8/32.0 26.1/31.8
//   workgroups      128                256               512
//   FP64            11.0/20.2 8.4/11.9 13.6/25.3 10.5/15.1 22.8/30.1 21.5/26.2
// Past that the chip is full and its waves only more: FP32 2304 to 4096 workgroups 0.94 to 0.98
// times as fast with three lattices (alone 0.95 to 1.21), FP64 768 36.2 / 37.9 alone.
static int deo_split_groups(const Geo& g) { return (int)(((g.V >> 1) + split::SITES - 1) / split::SITES); }
static bool deo_split_pays(const Geo& g, int set, bool fp64) {
  const int n = deo_split_groups(g);
  if (set == 3 || (g.V >> 1) >= (1 << 20)) return false;
  return n <= (fp64 ? 512 : 1280);
}

template <typename S, int RED>
static void deo_launch(const Geo& g, int nl, int pe, int set, int dag, int clv, int mode, typename Store<S>::R fac, S* out,
                       const S* in, const S* in0, const S* U, const S* C, const S* z, double* part, hipStream_t st) {
  const long long Vh = g.V >> 1;
  dim3 grid((unsigned)((Vh + EO_THREADS - 1) / EO_THREADS)), block(EO_THREADS);
  const bool sp = deo_split_pays(g, set, sizeof(S) == 8);
  if (sp) grid = dim3(deo_split_groups(g));
  const bool nt = (double)g.V * sizeof(S) * (4 * nl + 36 + 24) > DEO_STREAM_BYTES;
  const EoGeo eg = {{g.L[0], g.L[1], g.L[2], g.L[3]}, g.tbc, g.xcd_remap, g.V};
#define DEO_ARGS pe, set, clv, mode, fac, out, in, in0, U, C, z, part
#define DEO(NL, DAG)                                                                                                 \
  do {                                                                                                               \
    if (sp)                                                                                                          \
      hipLaunchKernelGGL((k_deo_split<S, NL, DAG, RED>), grid, block, 0, st, eg, 2.0f / g.L[0], 1.0f / g.L[1],        \
                         1.0f / g.L[2], DEO_ARGS);                                                                   \
    else if (nt) hipLaunchKernelGGL((k_deo<S, NL, DAG, true, RED>), grid, block, 0, st, eg, DEO_ARGS);                \
    else hipLaunchKernelGGL((k_deo<S, NL, DAG, false, RED>), grid, block, 0, st, eg, DEO_ARGS);                       \
  } while (0)
  if constexpr (RED != DEO_STORE) {
    if (nl != 18 || dag || set != 0 || mode != 2) throw std::logic_error("deo_launch: sums with the FP64 operator only");
    DEO(18, false);
  } else if (sizeof(S) == 4 && nl == 12) {
    if constexpr (std::is_same<S, float>::value) {
      if (dag) DEO(12, true);
      else DEO(12, false);
    }
  } else {
    if (dag) DEO(18, true);
    else DEO(18, false);
  }
#undef DEO
#undef DEO_ARGS
}

template <typename S>
void launch_deo(const Geo& g, int nl, int pe, int set, int dag, int clv, int mode, typename Store<S>::R fac, S* out,
                const S* in, const S* in0, const S* U, const S* C, hipStream_t st) {
  deo_launch<S, DEO_STORE>(g, nl, pe, set, dag, clv, mode, fac, out, in, in0, U, C, nullptr, nullptr, st);
}

int deo_reduce_groups(const Geo& g) {
  return deo_split_pays(g, 0, true) ? deo_split_groups(g) : (int)(((g.V >> 1) + EO_THREADS - 1) / EO_THREADS);
}
void launch_deo_reduce(const Geo& g, int pe, int red, double fac, double* out, const double* in, const double* in0,
                       const double* z, double* part, const double* U, const double* C, hipStream_t st) {
  if (red == DEO_DOT) deo_launch<double, DEO_DOT>(g, 18, pe, 0, 0, 1, 2, fac, out, in, in0, U, C, z, part, st);
  else deo_launch<double, DEO_NORM_DOT>(g, 18, pe, 0, 0, 1, 2, fac, out, in, in0, U, C, nullptr, part, st);
}

// ---------------------------------------------------------------- host layouts
// layout 0 (plain, x-compressed): spinor [Vh][24], links [2][4][Vh][18], clover [2][Vh][72].
// layout 1 (QWS AoSoA read as parity halves, qws.h:111-192 with deo_in_d.cc:65-90):
// vector i = xh/vlen + nxv (y + ny (z + nz t)), lane j = xh % vlen; spinor
// [(i*24 + k)*vlen + j], links glud[((i + vol*mu + 4*vol*p)*18 + k)*vlen + j], clover
// clvd[((i + vol*p)*72 + k)*vlen + j], vol = Vh / vlen.
__device__ __forceinline__ long long eo_host_offset(const Geo& g, int layout, int vlen, int kind, int p, int mu,
                                                    long long h, int k) {
  const long long Vh = g.V >> 1;
  if (layout == 0) {
    if (kind == 0) return h * 24 + k;
    if (kind == 1) return (((long long)p * 4 + mu) * Vh + h) * 18 + k;
    return ((long long)p * Vh + h) * 72 + k;
  }
  const long long vol = Vh / vlen;
  const long long i = h / vlen, j = h % vlen;  // xh = h % nxh and nxh % vlen == 0, so this splits xh
  if (kind == 0) return (i * 24 + k) * vlen + j;
  if (kind == 1) return ((i + vol * mu + 4 * vol * p) * 18 + k) * vlen + j;
  return ((i + vol * p) * 72 + k) * vlen + j;
}

// device offset (in reals) of real k: spinor/clover in 4-real (FP32) or 2-real
// (FP64) vectors, links in complex pairs
template <typename S>
__device__ __forceinline__ long long eo_dev_offset(const Geo& g, int kind, int nl, int p, int mu, long long h, int k) {
  const long long Vh = g.V >> 1;
  const int w = sizeof(S) == 8 ? 2 : 4;
  if (kind == 0) return ((long long)(k / w) * Vh + h) * w + (k % w);
  if (kind == 1) return ((((long long)p * 4 + mu) * (nl / 2) + (k >> 1)) * Vh + h) * 2 + (k & 1);
  return (((long long)p * (72 / w) + k / w) * Vh + h) * w + (k % w);
}

template <typename S>
__global__ void k_eo_import(Geo g, int kind, int layout, int vlen, int nl, const void* src, int src_is_double, S* dst) {
  const long long Vh = g.V >> 1;
  const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  const int np = kind == 0 ? 1 : 2;
  if (t >= Vh * np) return;
  const int p = (int)(t / Vh);
  const long long h = t - p * Vh;
  const int nmu = kind == 1 ? 4 : 1;
  const int nrec = kind == 0 ? 24 : (kind == 1 ? nl : 72);
  for (int mu = 0; mu < nmu; ++mu)
    for (int k = 0; k < nrec; ++k) {
      const long long o = eo_host_offset(g, layout, vlen, kind, p, mu, h, k);
      const double v = src_is_double ? ((const double*)src)[o] : (double)((const float*)src)[o];
      dst[eo_dev_offset<S>(g, kind, nl, p, mu, h, k)] = (S)v;
    }
}

template <typename S>
__global__ void k_eo_export(Geo g, int layout, int vlen, const S* src, void* dst, int dst_is_double) {
  const long long Vh = g.V >> 1;
  const long long h = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (h >= Vh) return;
  for (int k = 0; k < 24; ++k) {
    const long long o = eo_host_offset(g, layout, vlen, 0, 0, 0, h, k);
    const double v = (double)src[eo_dev_offset<S>(g, 0, 0, 0, 0, h, k)];
    if (dst_is_double) ((double*)dst)[o] = v;
    else ((float*)dst)[o] = (float)v;
  }
}

// Even/odd links and clover from the blocked-layout fields: the parity-p site h is
// the lattice site (2 xh + (p + y + z + t) % 2, y, z, t) (even extents only).
template <typename S>
__global__ void k_eo_gather(Geo g, int nl, const S* Ud, const S* Cd, S* Ue, S* Ce) {
  const long long Vh = g.V >> 1;
  const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (t >= 2 * Vh) return;
  const int p = (int)(t / Vh);
  const long long h = t - p * Vh;
  EoSite e;
  eo_coords(g, p, h, e);
  const int x[4] = {2 * e.c[0] + e.ick, e.c[1], e.c[2], e.c[3]};
  int bb[4], ll[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    bb[m] = x[m] / g.B[m];
    ll[m] = x[m] - bb[m] * g.B[m];
  }
  const long long s = site_index(g, bb, ll);
  const int nc = nl / 2;
  for (int mu = 0; mu < 4; ++mu)
    for (int k = 0; k < nc; ++k)
      for (int ri = 0; ri < 2; ++ri)
        Ue[((((long long)p * 4 + mu) * nc + k) * Vh + h) * 2 + ri] = Ud[(((long long)mu * nc + k) * g.V + s) * 2 + ri];
  const int w = sizeof(S) == 8 ? 2 : 4;
  for (int f = 0; f < 72 / w; ++f)
    for (int q = 0; q < w; ++q)
      Ce[(((long long)p * (72 / w) + f) * Vh + h) * w + q] = Cd[((long long)f * g.V + s) * w + q];
}

template <typename S>
void launch_eo_import(const Geo& g, int kind, int layout, int vlen, int nl, const void* src, int src_is_double, S* dst,
                      hipStream_t st) {
  const long long n = (g.V >> 1) * (kind == 0 ? 1 : 2);
  hipLaunchKernelGGL((k_eo_import<S>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, g, kind, layout, vlen, nl,
                     src, src_is_double, dst);
}
template <typename S>
void launch_eo_export(const Geo& g, int layout, int vlen, const S* src, void* dst, int dst_is_double, hipStream_t st) {
  const long long n = g.V >> 1;
  hipLaunchKernelGGL((k_eo_export<S>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, g, layout, vlen, src, dst,
                     dst_is_double);
}
template <typename S>
void launch_eo_gather(const Geo& g, int nl, const S* Ud, const S* Cd, S* Ue, S* Ce, hipStream_t st) {
  const long long n = g.V;
  hipLaunchKernelGGL((k_eo_gather<S>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, g, nl, Ud, Cd, Ue, Ce);
}

#define INST_EO(S)                                                                                                  \
  template void launch_deo<S>(const Geo&, int, int, int, int, int, int, typename Store<S>::R, S*, const S*,          \
                              const S*, const S*, const S*, hipStream_t);                                            \
  template void launch_eo_import<S>(const Geo&, int, int, int, int, const void*, int, S*, hipStream_t);              \
  template void launch_eo_export<S>(const Geo&, int, int, const S*, void*, int, hipStream_t);                        \
  template void launch_eo_gather<S>(const Geo&, int, const S*, const S*, S*, S*, hipStream_t);
INST_EO(float)
INST_EO(double)

}  // namespace qws
