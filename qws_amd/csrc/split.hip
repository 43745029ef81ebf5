// split.hip -- the hopping-term operators of dslash.hip for launches on few sites: four
// waves per 64 sites, and two block selections in one launch.
//
// A launch on few sites is one chain of latencies: site index, gathers, eight hops of
// about 120 vector instructions (a wave alone on its SIMD issues one every 4 to 5
// cycles), clover, store, on a fraction of the 256 CUs.  Here lane = site, and wave mu
// of the workgroup does the two hops of direction mu, both gathers in flight at once.
// The half spinors meet in LDS; each wave sums them and applies half the rows of one
// chirality of T^-1, loaded before the hops' arithmetic; waves 0 to 2 store one colour
// each.  Sums are taken in the order of hop_sum: bit for bit the results of k_hop.
#include <stdexcept>

#include "split_device.h"

namespace qws {

using namespace split;

namespace {

// What the kernel takes of Geo, and all its arguments in one, with a second operator only
// where there is one: a launch copies them, and the kernel's first loads fetch them from
// the host (Geo and two operators each time / so: D on 8^4, FP32, 3.44 / 3.34 us a call with
// three lattices in turn, 5.31 / 5.24 with one).
struct SplitGeo {
  int B[4], NB[4], sB[4], sN[4];
  int Vb, tbc, hopmask, xcd_remap;
  long long V;
};
template <typename S, bool PAIR> struct SplitArgs {
  SplitGeo g;
  float rb[3];
  int wg_per_blk;
  long long stride;
  const int* active;
  const S *U, *C;
  SplitPart<S> p[PAIR ? 2 : 1];
};

// The two hops of wave MU: half spinors into lh, zero for a hop that is not taken.
// rest() loads the clover.  FP64: a hop at a time, there are no registers for both.
template <typename S, int NL, int MU, typename Rest>
__device__ __forceinline__ void two_hops(const SplitGeo& g, int s, int first, const int b[4], const int l[4], bool on, int set,
                                         int mask, const S* in, const S* U,
                                         Cx<typename Store<S>::R> (*lh)[6][SITES], Rest&& rest) {
  using R = typename Store<S>::R;
  constexpr int NC = NL / 2, BOTH = sizeof(S) == 8 ? 0 : 1;
  const int lane = threadIdx.x & 63;
  Cx<R> v[1 + BOTH][12], u[1 + BOTH][9];
  bool take[2];
  auto load = [&](int d) {
    const int dir = d == 0 ? 1 : -1, ln = l[MU] + dir;
    const bool inside = ln >= 0 && ln < g.B[MU];
    const int bn = b[MU] + dir < 0 ? g.NB[MU] - 1 : b[MU] + dir >= g.NB[MU] ? 0 : b[MU] + dir;
    const int in_step = dir * g.sB[MU], out_step = in_step * (1 - g.B[MU]) + (bn - b[MU]) * g.sN[MU] * g.Vb;
    take[d] = on && (set == HOPS_INSIDE ? inside : ((mask >> (2 * MU + d)) & 1) && (set == HOPS_ALL || !inside));
    if (!__any(take[d])) return;
    // a lane without the hop reads the workgroup's first site: no traffic, no branch
    const unsigned n = take[d] ? s + (inside ? in_step : out_step) : first, at = d == 0 ? (take[d] ? s : first) : n;
#pragma unroll
    for (int j = 0; j < 6; ++j) IO<S>::load2(in, j, g.V, n * IO<S>::Q, v[d * BOTH] + 2 * j);
#pragma unroll
    for (int k = 0; k < NC; ++k) u[d * BOTH][k] = IO<S>::link(U, MU * NC + k, g.V, at * LINK_BYTES<S>);
  };
  auto hop = [&](int d) {
    Cx<R> h[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) h[k] = {0, 0};
    if (__any(take[d])) {
      Cx<R> a[6], m[6];
      if (NL == 12) link_row2(u[d * BOTH]);
      if (d == 0) {
        project<R, MU, +1>(v[d * BOTH], a);
        link_mult<R, +1>(u[d * BOTH], a, m);
      } else {
        project<R, MU, -1>(v[d * BOTH], a);
        link_mult<R, -1>(u[d * BOTH], a, m);
      }
#pragma unroll
      for (int k = 0; k < 6; ++k) h[k] = {take[d] ? m[k].re : R(0), take[d] ? m[k].im : R(0)};
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) lh[2 * MU + d][k][lane] = h[k];
  };
  // (the four waves' branches are not merged: that would hold their registers apart)
  asm volatile("; hops of direction %0" ::"i"(MU));
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

template <typename S, int NL, bool PAIR>
__global__ void __launch_bounds__(256) k_split(SplitArgs<S, PAIR> args) {
  using R = typename Store<S>::R;
  __shared__ Cx<R> lh[8][6][SITES];
  __shared__ Cx<R> ly[12][SITES];
  const SplitGeo& g = args.g;
  if (args.active && !args.active[blockIdx.y]) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const SplitPart<S>&p0 = args.p[0], &p1 = args.p[PAIR ? 1 : 0];
  const int wg_per_blk = args.wg_per_blk, n0 = PAIR ? p0.sel.n * wg_per_blk : (int)gridDim.x;
  const bool second = PAIR && (int)blockIdx.x >= n0;
  const int wg = second ? xcd_remap_n(g.xcd_remap, blockIdx.x - n0, gridDim.x - n0) : xcd_remap_n(g.xcd_remap, blockIdx.x, n0);
  const int* list = second ? p1.sel.list : p0.sel.list;
  const int set = second ? p1.set : p0.set, mask = g.hopmask & (second ? p1.mask : p0.mask);
  const R gamma = second ? p1.gamma : p0.gamma;
  S* out = second ? p1.out : p0.out;
  const S* ta = second ? p1.a : p0.a;
  const S* tb = second ? p1.b : p0.b;
  const S* tc = second ? p1.c : p0.c;
  const S* in = second ? p1.in : p0.in;
  const S* __restrict__ U = args.U;
  const S* __restrict__ C = args.C;
  const int bi = wg / wg_per_blk, blk = list ? list[bi] : bi;
  const int loc0 = (wg - bi * wg_per_blk) * SITES;
  const int loc = loc0 + lane < g.Vb ? loc0 + lane : loc0;
  bool on = loc0 + lane < g.Vb;
  const int base = blk * g.Vb, s = base + loc, first = base + loc0;
  int b[4], l[4], rem = blk;
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    b[m] = rem % g.NB[m];
    rem /= g.NB[m];
  }
  b[3] = rem;
  // loc / B by the reciprocal: exact below 2^20
  {
    const int q0 = (int)((loc + 0.5f) * args.rb[0]), q1 = (int)((q0 + 0.5f) * args.rb[1]), q2 = (int)((q1 + 0.5f) * args.rb[2]);
    l[0] = loc - q0 * g.B[0], l[1] = q0 - q1 * g.B[1], l[2] = q1 - q2 * g.B[2], l[3] = q2;
  }
  if (set == HOPS_FACE && out == ta && !tb && !tc) {  // sites without a face hop keep out
    bool face = false;
#pragma unroll
    for (int m = 0; m < 4; ++m) face |= (l[m] == 0) | (l[m] == g.B[m] - 1);
    on = on && face;
  }
  const unsigned sa = on ? s : first;
  const R tf_hi = b[3] == g.NB[3] - 1 && l[3] == g.B[3] - 1 ? R(2 * g.tbc) : R(2);
  const R tf_lo = b[3] == 0 && l[3] == 0 ? R(2 * g.tbc) : R(2);

  const long long off = blockIdx.y * args.stride;
  R ca[36];  // chirality wave & 1 of T^-1
  auto rest = [&]() { IO<S>::chir(C, wave & 1, g.V, sa * IO<S>::Q, ca); };
  const S* src = in + off;
  if (wave == 0) two_hops<S, NL, 0>(g, s, first, b, l, on, set, mask, src, U, lh, rest);
  else if (wave == 1) two_hops<S, NL, 1>(g, s, first, b, l, on, set, mask, src, U, lh, rest);
  else if (wave == 2) two_hops<S, NL, 2>(g, s, first, b, l, on, set, mask, src, U, lh, rest);
  else two_hops<S, NL, 3>(g, s, first, b, l, on, set, mask, src, U, lh, rest);
  __syncthreads();
  Cx<R> acc[12];
#pragma unroll
  for (int k = 0; k < 12; ++k) acc[k] = {0, 0};
  Cx<R> h[6];
#define ADD(MU, DIR, TF)                                                        \
  _Pragma("unroll") for (int k = 0; k < 6; ++k) h[k] = lh[2 * MU + (DIR < 0)][k][lane]; \
  reconstruct<R, MU, DIR>(h, TF, acc);
  ADD(0, +1, R(2)) ADD(0, -1, R(2)) ADD(1, +1, R(2)) ADD(1, -1, R(2))
  ADD(2, +1, R(2)) ADD(2, -1, R(2)) ADD(3, +1, tf_hi) ADD(3, -1, tf_lo)
#undef ADD
  Cx<R> x[6], y[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if (wave & 1) x[c] = csub(acc[c * 4], acc[c * 4 + 2]), x[3 + c] = csub(acc[c * 4 + 1], acc[c * 4 + 3]);
    else x[c] = cadd(acc[c * 4], acc[c * 4 + 2]), x[3 + c] = cadd(acc[c * 4 + 1], acc[c * 4 + 3]);
  }
  // wave c < 3 stores colour c; its terms a + b - c of the output
  Cx<R> v[2][2] = {};
  if (wave < 3) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      Cx<R> t[2];
      if (ta) IO<S>::load2(ta + off, 2 * wave + j, g.V, sa * IO<S>::Q, v[j]);
      if (tb) {
        IO<S>::load2(tb + off, 2 * wave + j, g.V, sa * IO<S>::Q, t);
        v[j][0] = cadd(v[j][0], t[0]), v[j][1] = cadd(v[j][1], t[1]);
      }
      if (tc) {
        IO<S>::load2(tc + off, 2 * wave + j, g.V, sa * IO<S>::Q, t);
        v[j][0] = csub(v[j][0], t[0]), v[j][1] = csub(v[j][1], t[1]);
      }
    }
  }
  if (wave < 2) herm3_mult<0>(ca, x, y);
  else herm3_mult<1>(ca, x, y);
#pragma unroll
  for (int k = 0; k < 3; ++k) ly[(wave & 1) * 6 + (wave >> 1) * 3 + k][lane] = y[k];
  __syncthreads();
  if (wave < 3 && on) {
    const Cx<R> y0 = ly[wave][lane], y1 = ly[3 + wave][lane], z0 = ly[6 + wave][lane], z1 = ly[9 + wave][lane];
    const Cx<R> t[2][2] = {{cadd(y0, z0), cadd(y1, z1)}, {csub(y0, z0), csub(y1, z1)}};
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      Cx<R> o[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) o[k] = {fmar(gamma, t[j][k].re, v[j][k].re), fmar(gamma, t[j][k].im, v[j][k].im)};
      IO<S>::store2(out + off, 2 * wave + j, g.V, (unsigned)s * IO<S>::Q, o);
    }
  }
}

}  // namespace

static long long split_groups(const Geo& g, long long sites, int nrhs) {
  return sites / g.Vb * ((g.Vb + SITES - 1) / SITES) * nrhs;
}
static bool split_fits(const Geo& g) { return g.Vb < (1 << 20) && g.V < (1 << 28); }

// The four waves shorten a launch that has the chip for itself; where launches of several
// streams share it, or one fills it, they are more waves for the same work.  So this kernel
// has the sizes at which it is no slower with three lattices on a stream each in turn, if one
// again and again, its fields in the caches, does not lose as much: us in turn / again and
// again, first k_hop, k_dslash or the staged kernels, then this one, by workgroups:
//   full operator, 4^4 blocks  FP32 12-real 512 6.3/13.9 4.4/7.2   1792 13.4/20.6 13.3/18.2   2560 21.8/26.0 24.5/24.1
//                              18-real 1792 16.3/21.4 16.1/19.6   2560 25.7/28.1 28.1/25.6
//                              FP64 256 7.6/15.6 4.5/6.9   448 8.8/18.8 7.3/10.7   512 9.5/19.0 9.9/13.8
//   (times as fast)  x halves  FP32 18-real 720 0.97/1.20, 1024 1.13/0.92, 1664 1.22/0.88, 2560 1.13/1.10, 4000 1.02/1.17
//                              12-real 720 0.94/1.30, 1024 1.05/1.02, 2592 1.03/1.03, 4000 0.96/1.05
//                              FP64 720 1.01/0.98, 1024 1.12/0.95, 1152 1.20/1.06, 2048 1.13/1.22, 10368 1.05/1.21
//   inside, a colour  halves   FP32 18-real 2000 1.05/0.95, 4320 0.97/1.17   12-real 512 1.08/1.3, 1024 0.95/0.97,
//                              2000 0.95/0.92   FP64 3000 0.98/1.08, 4320 0.96/1.13
//                    4^4       FP32 512 1.2/1.4, 768 0.87/1.2   FP64 768 1.13/1.02, 3456 1.02/1.13
//   faces, a colour  halves    FP32 360 1.06/1.37, 512 1.0/1.4, 1024 0.89/0.97   FP64 360 0.99/1.44, 512 0.81/1.25
//   (there most waves of k_hop have no face and leave at once)
// FP64 has two workgroups per CU (61 KB of LDS): past 448 a second round begins, nearly
// empty.  Blocks under 64 sites pay with idle lanes (2^4 blocks, 16384 workgroups: 90 / 100 us
// alone).  Several right-hand sides share links and clover in k_hop's loop, here only through
// the caches, but fill the chip better: solves of 3 on 32 12^2 10 by halves (1080 groups a
// colour) are 1.72 times as fast, with the limits of a single one 1.11 times.
bool split_pays(const Geo& g, int set, int sites, int nrhs, bool fp64, int nl) {
  if (set == HOPS_NONE || !split_fits(g)) return false;
  const long long wg = split_groups(g, sites, nrhs);
  const bool all = set == HOPS_ALL, b256 = g.Vb == 256;
  if (nrhs > 1) return wg <= (set == HOPS_FACE || g.Vb < SITES ? 1024 : 2048) && !(fp64 && all && wg > 512 && wg < 1024);
  if (wg <= (fp64 ? 448 : 512)) return true;
  if (set == HOPS_FACE || g.Vb < SITES) return false;
  if (fp64) return all ? !b256 && wg >= 1024 && wg <= 16384 : wg <= 3072;
  if (all) return b256 ? wg <= 1792 : wg >= 1024 && wg <= (nl == 12 ? 2592 : 4096);
  return !b256 && wg <= (nl == 12 ? 768 : 2048);
}
// Two operators in one launch, which is worth more: prec_ddd by halves (nsap 4, nm 2), two
// launches / one, 2048 groups in both: 12-real 1.05/1.05 and 1.02/1.13 times as fast as before
// there was either, 18-real 1.08/1.09 and 1.05/1.17.
bool split_pair_pays(const Geo& g, int sites, int nrhs) { return split_fits(g) && split_groups(g, sites, nrhs) <= 2048; }

template <typename S, int NL>
void launch_split(const Geo& g, const SplitPart<S>& p0, const SplitPart<S>& p1, const Batch& B, const S* U, const S* C,
                  hipStream_t st) {
  if (g.Vb >= (1 << 20) || g.V >= (1 << 28)) throw std::logic_error("launch_split: Vb < 2^20 and V < 2^28 sites");
  const int wpb = (g.Vb + SITES - 1) / SITES;
  const int n = (p0.sel.n + p1.sel.n) * wpb;
  if (n == 0) return;
  SplitArgs<S, true> args;
  for (int m = 0; m < 4; ++m) args.g.B[m] = g.B[m], args.g.NB[m] = g.NB[m], args.g.sB[m] = g.sB[m], args.g.sN[m] = g.sN[m];
  args.g.Vb = g.Vb, args.g.tbc = g.tbc, args.g.hopmask = g.hopmask, args.g.xcd_remap = g.xcd_remap, args.g.V = g.V;
  for (int m = 0; m < 3; ++m) args.rb[m] = 1.0f / g.B[m];
  args.wg_per_blk = wpb, args.stride = B.stride, args.active = B.active, args.U = U, args.C = C;
  args.p[0] = p0, args.p[1] = p1;
  if (p1.sel.n) {
    hipLaunchKernelGGL((k_split<S, NL, true>), dim3(n, B.n), dim3(256), 0, st, args);
  } else {
    const SplitArgs<S, false> one = {args.g, {args.rb[0], args.rb[1], args.rb[2]}, wpb, B.stride, B.active, U, C, {p0}};
    hipLaunchKernelGGL((k_split<S, NL, false>), dim3(n, B.n), dim3(256), 0, st, one);
  }
}

#define INST_SPLIT(S, NL)                                                                                            \
  template void launch_split<S, NL>(const Geo&, const SplitPart<S>&, const SplitPart<S>&, const Batch&, const S*, const S*, \
                                    hipStream_t);
INST_SPLIT(float, 18)
INST_SPLIT(float, 12)
INST_SPLIT(double, 18)
INST_SPLIT(__half, 18)
INST_SPLIT(__half, 12)

}  // namespace qws
