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

// The two hops of wave MU: half spinors into lh, zero for a hop that is not taken.
// rest() loads the clover.  FP64: a hop at a time, there are no registers for both.
template <typename S, int NL, int MU, typename Rest>
__device__ __forceinline__ void two_hops(const Geo& g, int s, int first, const int b[4], const int l[4], bool on, int set,
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

template <typename S, int NL>
__global__ void __launch_bounds__(256)
k_split(Geo g, SplitPart<S> p0, SplitPart<S> p1, float rb0, float rb1, float rb2, int wg_per_blk, long long stride,
        const int* __restrict__ active, const S* __restrict__ U, const S* __restrict__ C) {
  using R = typename Store<S>::R;
  __shared__ Cx<R> lh[8][6][SITES];
  __shared__ Cx<R> ly[12][SITES];
  if (active && !active[blockIdx.y]) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = p0.sel.n * wg_per_blk;
  const bool second = (int)blockIdx.x >= n0;
  const int wg = second ? xcd_remap(g, blockIdx.x - n0, gridDim.x - n0) : xcd_remap(g, blockIdx.x, n0);
  const int* list = second ? p1.sel.list : p0.sel.list;
  const int set = second ? p1.set : p0.set, mask = g.hopmask & (second ? p1.mask : p0.mask);
  const R gamma = second ? p1.gamma : p0.gamma;
  S* out = second ? p1.out : p0.out;
  const S* ta = second ? p1.a : p0.a;
  const S* tb = second ? p1.b : p0.b;
  const S* tc = second ? p1.c : p0.c;
  const S* in = second ? p1.in : p0.in;
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
    const int q0 = (int)((loc + 0.5f) * rb0), q1 = (int)((q0 + 0.5f) * rb1), q2 = (int)((q1 + 0.5f) * rb2);
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

  const long long off = blockIdx.y * stride;
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

// Times in us, k_hop, k_dslash or the staged kernels / this one, on 18-real links:
//   full operator    8^4 (64 workgroups)  FP32 12.2 / 5.5  FP64 15.3 / 6.4
//                    16^4, 4^4 blocks (1024)   16.3 / 13.1      24.2 / 23.0
//                    16^2 32^2, 4^4 blocks (4096) 43.2 / 40.6   98.5 / 98.2
//                    24^3 32, 4^4 blocks (6912) 78.3 / 80.0    163 / 163: to 4096
//                    16^3 8, 4^4 blocks (512)   14.5 / 7.7      19.1 / 13.0
//                    32 12^2 10, halves (720)  11.8 / 10.0      17.0 / 19.3
//                    48 24^3, halves (10368)   93.2 / 107        285 / 255: FP32 to 4096
//   inside           48 24^3, halves (5184)    59.4 / 50.6       129 / 117
//   (32^3 64 by halves is the same either way, by 4^4 blocks up to 8% slower here)
//   faces            16^4, 4^4 blocks (512)    12.7 / 7.5       16.7 / 12.7
//                    32 16^3, halves (1024)    11.5 / 12.6      17.6 / 19.7: to 1024
//   (there most waves of k_hop have no face and leave at once)
// FP64 has two workgroups per CU (61 KB of LDS): past 512 the second round is nearly
// empty, and the full operator goes back to k_dslash up to 1024.
// A block's last workgroup has idle lanes, which blocks under 64 sites pay for with more
// of them: to 1024 (2^4 blocks, 16384 workgroups: 90 / 100 us).  Right-hand sides share
// links and clover in k_hop's loop, here only through the caches: to 2048.
bool split_pays(const Geo& g, int set, int sites, int nrhs, bool fp64) {
  if (set == HOPS_NONE || g.Vb >= (1 << 20) || g.V >= (1 << 28)) return false;
  const long long wg = (long long)(sites / g.Vb) * ((g.Vb + SITES - 1) / SITES) * nrhs;
  if (set == HOPS_FACE || g.Vb < SITES) return wg <= 1024;
  if (fp64 && set == HOPS_ALL && wg > 512 && wg < 1024) return false;
  if (nrhs > 1) return wg <= 2048;
  return wg <= (set == HOPS_ALL && (g.Vb == 256 || !fp64) ? 4096 : 16384);
}

template <typename S, int NL>
void launch_split(const Geo& g, const SplitPart<S>& p0, const SplitPart<S>& p1, const Batch& B, const S* U, const S* C,
                  hipStream_t st) {
  if (g.Vb >= (1 << 20) || g.V >= (1 << 28)) throw std::logic_error("launch_split: Vb < 2^20 and V < 2^28 sites");
  const int wpb = (g.Vb + SITES - 1) / SITES;
  const int n = (p0.sel.n + p1.sel.n) * wpb;
  if (n == 0) return;
  hipLaunchKernelGGL((k_split<S, NL>), dim3(n, B.n), dim3(256), 0, st, g, p0, p1, 1.0f / g.B[0], 1.0f / g.B[1], 1.0f / g.B[2],
                     wpb, B.stride, B.active, U, C);
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
