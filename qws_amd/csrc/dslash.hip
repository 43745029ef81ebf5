// dslash.hip -- hopping-term kernels: D, block-local D_in, face terms and the
// fused SAP updates, all as  out = a + b - c + gamma * T^-1 H_set(in).
//
// Reference semantics: ddd_in_s.cc:72-374 / ddd_in_d.cc:66-196 (hops inside a
// domain, then T^-1, then out = in - kappa * (...)), ddd_out_s.cc:112-626 and
// ddd_out_d.cc:84-235 (face hops of a domain, T^-1, out += factor * (...)),
// qws.cc:625-644 (full operator).  On one GPU the faces are read in place from
// the neighbouring block instead of being packed and exchanged.
#include <algorithm>
#include <type_traits>

#include "kernels.h"

namespace qws {

constexpr int HOP_THREADS = 256;

// Whether the full operator reads its clover and writes its output past the caches (NT).
// Up to about the last-level cache's 256 MB the operator's data come from there the next
// time; above, they only push out spinors and links that neighbouring blocks read again
// (32^3x64 by 4^4 blocks: 1.47 times the bytes needed came from beyond L2).  us with
// ordinary / nontemporal accesses, 4^4 blocks, FP32 unless said:
//   198 MB  43.0 / 46.7    226 MB  48.0 / 51.7    264 MB  54.9 / 55.2    297 MB  64.5 / 61.0
//   340 MB  77.3 / 69.0    446 MB   108 / 88.9   1409 MB   337 / 313     FP64 1019 MB 253 / 235
constexpr double DSLASH_STREAM_BYTES = 280e6;

// Blocks that an XCD takes in turn in the LDS-staged full operators (xcd_remap_chunked), in index
// order, above DSLASH_STREAM_BYTES.  With a contiguous eighth of the lattice for each XCD
// every face that its L2 has lost comes from memory; side by side the XCDs find it in the
// last-level cache.  us, a contiguous range / chunks of 8 / of 64:
//   FP64  24^3 48 234 / 214 / 221   32^4 364 / 353 / 348   40 24 32 40 444 / 404 / 412   32^3 64 768 / 681 / 721
//   FP32  24^3 48  94 /  93 /  93   32^4 152 / 158 / 150   40 24 32 40 187 / 178 / 179   32^3 64 321 / 310 / 313
// (No gain for k_dslash on large blocks, nor for the even/odd operator.)  Below that an
// operator on fields that it has just had finds more of its own range in its L2, and on
// few blocks the chunks fill the XCDs unevenly.  Three lattices in turn / one again and
// again, contiguous ranges and chunks:
//   FP32  16^3 24 11.7 / 19.8 and 14.5 / 21.2   24^4 50.5 / 49.4 and 50.2 / 52.3
//   FP64  8^2 16 56 16.3 / 22.7 and 16.9 / 23.2   16^3 40 55.7 / 62.0 and 55.3 / 59.7
constexpr int DSLASH_CHUNK_64 = 8, DSLASH_CHUNK_32 = 64;

template <typename S, int NL, int SET>
__global__ void __launch_bounds__(HOP_THREADS)
k_hop(Geo g, const int* __restrict__ list, int wg_per_blk, int nrhs, long long stride, const int* __restrict__ active,
      typename Store<S>::R gamma, S* out, const S* a, const S* b, const S* c, const S* __restrict__ in,
      const S* __restrict__ U, const S* __restrict__ C, int skip_interior) {
  using R = typename Store<S>::R;
  const int wg = xcd_remap(g, blockIdx.x, gridDim.x);
  const int bi = wg / wg_per_blk;
  const int blk = list ? list[bi] : bi;
  const int loc = (wg - bi * wg_per_blk) * HOP_THREADS + threadIdx.x;
  if (loc >= g.Vb) return;
  const long long s = (long long)blk * g.Vb + loc;
  SiteC sc;
  site_coords(g, s, sc);
  if ((SET == HOPS_FACE || SET == HOPS_FACE_MASKED) && skip_interior) {
    bool face = false;
#pragma unroll
    for (int m = 0; m < 4; ++m) face |= (sc.l[m] == 0) | (sc.l[m] == g.B[m] - 1);
    if (!face) return;
  }
  // right-hand sides share this thread's links and clover (cache-resident after the first)
  for (int r = 0; r < nrhs; ++r) {
    if (active && !active[r]) continue;
    const long long off = r * stride;
    const long long sr = opaque_v(s);
    SiteC scr;
    site_coords(g, sr, scr);
    Cx<R> acc[12];
    hop_sum<S, NL, SET>(g, sr, scr, in + off, opaque(U), acc);
    clover_apply<S>(opaque(C), sr, g.V, acc);
    Cx<R> v[12];
    if (a) {
      SpinorIO<S>::load(a + off, s, g.V, v);
    } else {
#pragma unroll
      for (int k = 0; k < 12; ++k) v[k] = {0, 0};
    }
    if (b) {
      Cx<R> w[12];
      SpinorIO<S>::load(b + off, s, g.V, w);
#pragma unroll
      for (int k = 0; k < 12; ++k) v[k] = cadd(v[k], w[k]);
    }
    if (c) {
      Cx<R> w[12];
      SpinorIO<S>::load(c + off, s, g.V, w);
#pragma unroll
      for (int k = 0; k < 12; ++k) v[k] = csub(v[k], w[k]);
    }
#pragma unroll
    for (int k = 0; k < 12; ++k) v[k] = {fmar(gamma, acc[k].re, v[k].re), fmar(gamma, acc[k].im, v[k].im)};
    SpinorIO<S>::store(out + off, s, g.V, v);
  }
}

// The right-hand side of logical workgroup wg of a full operator, by its offset in the
// spinors, and in wg the workgroup of its blocks; false where it is not active.  Those
// of one block are neighbours, on one XCD, so that the links and the clover inverse come
// from its L2 for all but the first (12 right-hand sides on 16^3 x 32, FP64, one after
// another / so: 680 / 393 us).
__device__ __forceinline__ bool rhs_of(int& wg, int nrhs, long long stride, const int* active, long long& off) {
  const int r = nrhs == 1 ? 0 : wg % nrhs;
  if (nrhs != 1) wg /= nrhs;
  off = r * stride;
  return !(active && !active[r]);
}

// Full operator out = in + gamma T^-1 H in over every site: the kernel for D itself
// (ddd_d_, ddd_s_ and the outer solver's D).  Written without the generality of k_hop
// (RHS loop, a/b/c terms, block lists) it keeps the live state of a thread small (about
// 90 VGPRs in FP32).  It is compiled for at most
// 3 waves per SIMD (amdgpu_waves_per_eu): the schedule that results orders the
// neighbour gathers so that FP32 32^3x64 fetches 1.3x less from HBM than the default
// schedule and runs 2% faster (the register count still admits 5 waves per SIMD).
template <typename S, int NL, bool NT>
__global__ void __launch_bounds__(HOP_THREADS) __attribute__((amdgpu_waves_per_eu(1, 3)))
k_dslash(Geo g, const int* __restrict__ order, int wg_per_blk, int nrhs, long long stride,
         const int* __restrict__ active, typename Store<S>::R gamma, S* __restrict__ out, const S* __restrict__ in,
         const S* __restrict__ U, const S* __restrict__ C) {
  using R = typename Store<S>::R;
  int wg = xcd_remap(g, blockIdx.x, gridDim.x);
  long long off;
  if (!rhs_of(wg, nrhs, stride, active, off)) return;
  in += off, out += off;
  const int bi = wg / wg_per_blk;
  const int loc = (wg - bi * wg_per_blk) * HOP_THREADS + threadIdx.x;
  if (loc >= g.Vb) return;
  const long long s = (long long)order[bi] * g.Vb + loc;
  SiteC sc;
  site_coords(g, s, sc);
  Cx<R> acc[12];
  hop_sum<S, NL, HOPS_ALL>(g, s, sc, in, U, acc);
  clover_apply<S, NT>(C, s, g.V, acc);
  Cx<R> v[12];
  SpinorIO<S>::load(in, s, g.V, v);
#pragma unroll
  for (int k = 0; k < 12; ++k) v[k] = {fmar(gamma, acc[k].re, v[k].re), fmar(gamma, acc[k].im, v[k].im)};
  SpinorIO<S>::template store<NT>(out, s, g.V, v);
}

// One hop of the LDS-staged full operator: the neighbour's spinor from LDS when it
// lies in the block, from global memory across a block face.
template <int NL, int MU, int DIR>
__device__ __forceinline__ void hop_staged(const Geo& g, long long s, const SiteC& c, int t, const float4* lx,
                                           const float* in, const float* U, Cx<float> acc[12]) {
  if (!(g.hopmask & (1 << (2 * MU + (DIR > 0 ? 0 : 1))))) return;
  bool inside;
  const long long n = neighbour(g, s, c, MU, DIR, inside);
  Cx<float> v[12], a[6], b[6], u[9];
  if (inside) {
    const int tn = t + DIR * g.sB[MU];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      const float4 q = lx[j * HOP_THREADS + tn];
      v[2 * j] = {q.x, q.y};
      v[2 * j + 1] = {q.z, q.w};
    }
  } else {
    SpinorIO<float>::load(in, n, g.V, v);
  }
  project<float, MU, DIR>(v, a);
  load_link<float, NL>(U, MU, DIR > 0 ? s : n, g.V, u);
  link_mult<float, DIR>(u, a, b);
  float tf = 2.0f;
  if (MU == 3) {
    const int tt = c.b[3] * g.B[3] + c.l[3];
    if ((DIR > 0 && tt == g.L[3] - 1) || (DIR < 0 && tt == 0)) tf = 2.0f * g.tbc;
  }
  reconstruct<float, MU, DIR>(b, tf, acc);
}

// Full operator, FP32, one workgroup per 256-site block: the block's own spinor is
// loaded once with coalesced 128-bit loads and staged in LDS; the hops inside the
// block read it there, only the hops across a block face gather from global memory.
// Each block's spinor thus crosses L2 once for its own hops instead of up to nine
// times, and the neighbour requests left are the faces (FP32 32^3x64: 1.39x the
// algorithmic HBM bytes against 1.48x for k_dslash, 6% faster).  W is the number of
// waves per SIMD the compiler schedules for (amdgpu_waves_per_eu); at about 104
// VGPRs 4 waves are resident either way.
// (Nontemporal loads of the links were measured slower, with more L2 misses: the
// backward hops read them again.)
template <int NL, int W, bool NT>
__global__ void __launch_bounds__(HOP_THREADS) __attribute__((amdgpu_waves_per_eu(1, W)))
k_dslash_lds(Geo g, const int* __restrict__ order, int nrhs, long long stride, const int* __restrict__ active, float gamma, float* __restrict__ out,
             const float* __restrict__ in, const float* __restrict__ U, const float* __restrict__ C) {
  __shared__ float4 lx[6 * HOP_THREADS];
  int wg = xcd_remap_chunked(g, blockIdx.x, gridDim.x);
  long long off;
  if (!rhs_of(wg, nrhs, stride, active, off)) return;
  in += off, out += off;
  const int t = threadIdx.x;
  const long long s = (long long)order[wg] * HOP_THREADS + t;
  const float4* iv = reinterpret_cast<const float4*>(in);
#pragma unroll
  for (int j = 0; j < 6; ++j) lx[j * HOP_THREADS + t] = iv[(long long)j * g.V + s];
  __syncthreads();
  SiteC sc;
  site_coords(g, s, sc);
  Cx<float> acc[12];
#pragma unroll
  for (int k = 0; k < 12; ++k) acc[k] = {0, 0};
  hop_staged<NL, 0, +1>(g, s, sc, t, lx, in, U, acc);
  hop_staged<NL, 0, -1>(g, s, sc, t, lx, in, U, acc);
  hop_staged<NL, 1, +1>(g, s, sc, t, lx, in, U, acc);
  hop_staged<NL, 1, -1>(g, s, sc, t, lx, in, U, acc);
  hop_staged<NL, 2, +1>(g, s, sc, t, lx, in, U, acc);
  hop_staged<NL, 2, -1>(g, s, sc, t, lx, in, U, acc);
  hop_staged<NL, 3, +1>(g, s, sc, t, lx, in, U, acc);
  hop_staged<NL, 3, -1>(g, s, sc, t, lx, in, U, acc);
  clover_apply<float, NT>(C, s, g.V, acc);
  f4v* ov = reinterpret_cast<f4v*>(out);
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const float4 o = lx[j * HOP_THREADS + t];
    st_nt<NT>(ov + ((long long)j * g.V + s), f4v{fmar(gamma, acc[2 * j].re, o.x), fmar(gamma, acc[2 * j].im, o.y),
                                                 fmar(gamma, acc[2 * j + 1].re, o.z), fmar(gamma, acc[2 * j + 1].im, o.w)});
  }
}

template <int NL>
void launch_dslash_lds(const Geo& g, BlockSel sel, const Batch& B, bool nt, float gamma, float* out, const float* in,
                       const float* U, const float* C, hipStream_t st) {
#define DSL_LDS(W, NT)                                                                                             \
  hipLaunchKernelGGL((k_dslash_lds<NL, W, NT>), dim3(sel.n * B.n), dim3(HOP_THREADS), 0, st, g, sel.list, B.n, B.stride, \
                     B.active, gamma, out, in, U, C)
  if (g.dslash_kernel == 3) {
    if (nt) DSL_LDS(3, true);
    else DSL_LDS(3, false);
  } else {
    if (nt) DSL_LDS(4, true);
    else DSL_LDS(4, false);
  }
#undef DSL_LDS
}

// One FP64 hop of the LDS-staged full operator: the arithmetic of one_hop<double, 18>,
// the neighbour's spinor from LDS when it lies in the block.
template <int MU, int DIR>
__device__ __forceinline__ void hop_staged_d(const Geo& g, long long s, const SiteC& c, int t, const double2* lx,
                                             const double* in, const double* U, Cx<double> acc[12]) {
  if (!(g.hopmask & (1 << (2 * MU + (DIR > 0 ? 0 : 1))))) return;
  bool inside;
  const long long n = neighbour(g, s, c, MU, DIR, inside);
  Cx<double> v[12], a[6], b[6], u[9];
  if (inside) {
    const int tn = t + DIR * g.sB[MU];
#pragma unroll
    for (int k = 0; k < 12; ++k) {
      const double2 q = lx[k * HOP_THREADS + tn];
      v[k] = {q.x, q.y};
    }
  } else {
    SpinorIO<double>::load(in, n, g.V, v);
  }
  project<double, MU, DIR>(v, a);
  load_link<double, 18>(U, MU, DIR > 0 ? s : n, g.V, u);
  link_mult<double, DIR>(u, a, b);
  double tf = 2.0;
  if (MU == 3) {
    const int tt = c.b[3] * g.B[3] + c.l[3];
    if ((DIR > 0 && tt == g.L[3] - 1) || (DIR < 0 && tt == 0)) tf = double(2 * g.tbc);
  }
  reconstruct<double, MU, DIR>(b, tf, acc);
}

// FP64 full operator (the outer solver's D, ddd_d_) on 256-site blocks with the block's
// spinor staged in LDS (12 double2 planes, 48 KB): bit for bit k_dslash<double, 18>.
template <int W, bool NT>
__global__ void __launch_bounds__(HOP_THREADS) __attribute__((amdgpu_waves_per_eu(1, W)))
k_dslash_lds_d(Geo g, const int* __restrict__ order, int nrhs, long long stride, const int* __restrict__ active, double gamma,
               double* __restrict__ out, const double* __restrict__ in, const double* __restrict__ U,
               const double* __restrict__ C) {
  __shared__ double2 lx[12 * HOP_THREADS];
  int wg = xcd_remap_chunked(g, blockIdx.x, gridDim.x);
  long long off;
  if (!rhs_of(wg, nrhs, stride, active, off)) return;
  in += off, out += off;
  const int t = threadIdx.x;
  const long long s = (long long)order[wg] * HOP_THREADS + t;
  const double2* iv = reinterpret_cast<const double2*>(in);
#pragma unroll
  for (int k = 0; k < 12; ++k) lx[k * HOP_THREADS + t] = iv[(long long)k * g.V + s];
  __syncthreads();
  SiteC sc;
  site_coords(g, s, sc);
  Cx<double> acc[12];
#pragma unroll
  for (int k = 0; k < 12; ++k) acc[k] = {0, 0};
  hop_staged_d<0, +1>(g, s, sc, t, lx, in, U, acc);
  hop_staged_d<0, -1>(g, s, sc, t, lx, in, U, acc);
  hop_staged_d<1, +1>(g, s, sc, t, lx, in, U, acc);
  hop_staged_d<1, -1>(g, s, sc, t, lx, in, U, acc);
  hop_staged_d<2, +1>(g, s, sc, t, lx, in, U, acc);
  hop_staged_d<2, -1>(g, s, sc, t, lx, in, U, acc);
  hop_staged_d<3, +1>(g, s, sc, t, lx, in, U, acc);
  hop_staged_d<3, -1>(g, s, sc, t, lx, in, U, acc);
  clover_apply<double, NT>(C, s, g.V, acc);
  d2v* ov = reinterpret_cast<d2v*>(out);
#pragma unroll
  for (int k = 0; k < 12; ++k) {
    const double2 o = lx[k * HOP_THREADS + t];
    st_nt<NT>(ov + ((long long)k * g.V + s), d2v{fmar(gamma, acc[k].re, o.x), fmar(gamma, acc[k].im, o.y)});
  }
}

template <typename S, int NL>
void launch_hop(const Geo& g, BlockSel sel, const Batch& B, int set, typename Store<S>::R gamma, S* out, const S* a,
                const S* b, const S* c, const S* in, const S* U, const S* C, hipStream_t st, bool index_order) {
  const bool full = set == HOPS_ALL && sel.n == g.nblk && a == in && b == nullptr && c == nullptr && out != in;
  // a kernel that was asked for by name (qwsg_set_dslash_kernel, the environment) is the one that runs
  const bool named = full && g.Vb == HOP_THREADS &&
                     ((std::is_same<S, float>::value && g.dslash_kernel != DSLASH_AUTO) ||
                      (std::is_same<S, double>::value && g.dslash_kernel_d != DSLASH_AUTO));
  if (!named && split_pays(g, set, sel.n * g.Vb, B.n, std::is_same<S, double>::value, NL)) {
    SplitPart<S> p;
    p.sel = sel, p.set = set, p.gamma = gamma, p.out = out, p.a = a, p.b = b, p.c = c, p.in = in;
    launch_split<S, NL>(g, p, SplitPart<S>(), B, U, C, st);
    return;
  }
  if (full) {
    // the full operator (several right-hand sides share their clover through the caches)
    const int wpb = (g.Vb + HOP_THREADS - 1) / HOP_THREADS;
    // a grid has fewer than 2^32 work-items: 16 right-hand sides on 32^4 in blocks of one
    // site, a workgroup each, take two launches
    const int most = (int)std::max(1LL, ((1LL << 32) - 1) / ((long long)sel.n * wpb * HOP_THREADS));
    if (B.n > most) {
      for (int r = 0; r < B.n; r += most) {
        const Batch part{std::min(most, B.n - r), B.stride, B.active ? B.active + r : nullptr};
        launch_hop<S, NL>(g, sel, part, set, gamma, out + r * B.stride, in + r * B.stride, nullptr, nullptr,
                          in + r * B.stride, U, C, st, index_order);
      }
      return;
    }
    const bool nt = B.n == 1 && operator_bytes<S>(g, NL) > DSLASH_STREAM_BYTES;
    Geo gc = g;
    if (index_order && nt) gc.xcd_chunk = sizeof(S) == 8 ? DSLASH_CHUNK_64 : DSLASH_CHUNK_32;
    if constexpr (std::is_same<S, float>::value) {
      if (g.Vb == HOP_THREADS && g.dslash_kernel != 0) {
        launch_dslash_lds<NL>(gc, sel, B, nt, gamma, out, in, U, C, st);
        return;
      }
    }
    if constexpr (std::is_same<S, double>::value && NL == 18) {
      if (g.Vb == HOP_THREADS && g.dslash_kernel_d != 0) {
#define DSL_LDS(W, NT)                                                                                          \
  hipLaunchKernelGGL((k_dslash_lds_d<W, NT>), dim3(sel.n * B.n), dim3(HOP_THREADS), 0, st, gc, sel.list, B.n, B.stride, \
                     B.active, gamma, out, in, U, C)
        if (g.dslash_kernel_d == 3) {
          if (nt) DSL_LDS(3, true);
          else DSL_LDS(3, false);
        } else {
          if (nt) DSL_LDS(2, true);
          else DSL_LDS(2, false);
        }
#undef DSL_LDS
        return;
      }
    }
#define DSL(NT)                                                                                                  \
  hipLaunchKernelGGL((k_dslash<S, NL, NT>), dim3(sel.n * wpb * B.n), dim3(HOP_THREADS), 0, st, g, sel.list, wpb, B.n, \
                     B.stride, B.active, gamma, out, in, U, C)
    if (nt) DSL(true);
    else DSL(false);
#undef DSL
    return;
  }
  const int wpb = (g.Vb + HOP_THREADS - 1) / HOP_THREADS;
  dim3 grid(sel.n * wpb), block(HOP_THREADS);
  const int skip = (set == HOPS_FACE && out == a && b == nullptr && c == nullptr) ? 1 : 0;
#define HOP_ARGS g, sel.list, wpb, B.n, B.stride, B.active, gamma, out, a, b, c, in, U, C
  switch (set) {
    case HOPS_ALL:
      hipLaunchKernelGGL((k_hop<S, NL, HOPS_ALL>), grid, block, 0, st, HOP_ARGS, skip);
      break;
    case HOPS_INSIDE:
      hipLaunchKernelGGL((k_hop<S, NL, HOPS_INSIDE>), grid, block, 0, st, HOP_ARGS, skip);
      break;
    case HOPS_FACE:
      if (g.hopmask == 0xFF) hipLaunchKernelGGL((k_hop<S, NL, HOPS_FACE>), grid, block, 0, st, HOP_ARGS, skip);
      else hipLaunchKernelGGL((k_hop<S, NL, HOPS_FACE_MASKED>), grid, block, 0, st, HOP_ARGS, skip);
      break;
    default:
      hipLaunchKernelGGL((k_hop<S, NL, HOPS_NONE>), grid, block, 0, st, HOP_ARGS, 0);
  }
#undef HOP_ARGS
}

#define INST_HOP(S, NL)                                                                                           \
  template void launch_hop<S, NL>(const Geo&, BlockSel, const Batch&, int, typename Store<S>::R, S*, const S*,     \
                                  const S*, const S*, const S*, const S*, const S*, hipStream_t, bool);
INST_HOP(float, 18)
INST_HOP(float, 12)
INST_HOP(double, 18)
INST_HOP(__half, 18)
INST_HOP(__half, 12)

}  // namespace qws
