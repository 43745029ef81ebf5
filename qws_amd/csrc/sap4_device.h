// sap4_device.h -- what the fused SAP kernels for 4^4 blocks share (sap4.hip, sap4h.hip):
// positions in LDS, half spinors, the face buffer's slots.
#pragma once

#include "kernels.h"
#include "sap.h"
#include "sap_device.h"

namespace qws {
namespace sap4 {

constexpr int VB = 256;  // sites per block = threads per workgroup
constexpr int FS = 512;  // face slots per block (sap_kernels.inc has their order)

// At most that many workgroups, a quarter of the CUs: the wide kernel.  It takes a CU for
// itself, so that launches of other streams have to find theirs.  us, the other / it: 8 blocks
// (8^4) nm 2 16.7 / 14.6, nm 6 29.2 / 23.5; 64 blocks nm 6 31.6 / 26.1; 256 blocks nm 6 alone 34.8
// / 29.8, but nm 2 on three streams at once 11.7 / 17.5 a launch  FP16: 8 blocks nm 2 15.6 /
// 14.1, nm 6 26.3 / 22.7.
constexpr int WIDE_GROUPS = 64;

// Position of block site s = (x, y, z, t) in an LDS plane of float4: its low four bits
// (x, y) XORed by a constant for each z.  A 128-bit LDS read serves lanes 0-3, 12-15 and
// 20-27 (then the others of 32) at once from 16 groups of 16 bytes, a write eight lanes in
// a row from 8 groups; with these constants, and the lane order of link_site, every access
// of block_hops is free of bank conflicts.
__device__ __forceinline__ int lds_pos(int s) { return s ^ ((0x7AD0 >> ((s >> 2) & 12)) & 15); }

// The site with coordinate l along mu whose other coordinates are those of lane j, the
// first of them fastest (the order of the face slots).
__device__ __forceinline__ int slice_site(int mu, int l, int j) {
  if (mu == 0) return l + 4 * j;
  if (mu == 1) return (j & 3) + 4 * l + 16 * (j >> 2);
  if (mu == 2) return (j & 15) + 16 * l + 64 * (j >> 4);
  return j + 64 * l;
}
// The same for the links inside the block; along x the lane bits are y0 z0 z1 y1 t0 t1.
__device__ __forceinline__ int link_site(int mu, int l, int j) {
  return slice_site(mu, l, mu == 0 ? (j & 0x31) | ((j & 6) << 1) | ((j & 8) >> 2) : j);
}

// Nothing is scheduled across this: keeps LDS reads where they are issued, ahead of the
// arithmetic that hides their latency.
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }

__device__ __forceinline__ void store_half(f4v* lh, int mu, int p, const Cx<float> h[6]) {
#pragma unroll
  for (int k = 0; k < 3; ++k)
    lh[(mu * 3 + k) * VB + p] = f4v{h[2 * k].re, h[2 * k].im, h[2 * k + 1].re, h[2 * k + 1].im};
}

// The half spinors of the four directions at position p, and their sums into the site.
struct Halves {
  f4v q[4][3];
};
__device__ __forceinline__ void read_halves(const f4v* lh, int p, Halves& h) {
#pragma unroll
  for (int mu = 0; mu < 4; ++mu)
#pragma unroll
    for (int k = 0; k < 3; ++k) h.q[mu][k] = lh[(mu * 3 + k) * VB + p];
}
template <int MU, int DIR>
__device__ __forceinline__ void add_half(const Halves& hs, float tf, Cx<float> acc[12]) {
  Cx<float> h[6];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    h[2 * k] = {hs.q[MU][k].x, hs.q[MU][k].y};
    h[2 * k + 1] = {hs.q[MU][k].z, hs.q[MU][k].w};
  }
  reconstruct<float, MU, DIR>(h, tf, acc);
}

// The thread's index, as a value that the compiler computes anew where it is asked for:
// what derives from it (addresses, coordinates) is not kept in registers meanwhile.
__device__ __forceinline__ unsigned fresh_thread() {
  unsigned t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}
struct Coord {
  int x, y, z, t;
};
__device__ __forceinline__ Coord coord(unsigned t, int wave) {
  return {(int)(t & 3), (int)((t >> 2) & 3), (int)((t >> 4) & 3), wave};
}

// A wave's slots of the face update, direction MU = its own number: the + side's half
// spinors in q[0..2], the - side's in q[3..5].
__device__ __forceinline__ void read_slots(const f4v* slots, int wave, unsigned j, f4v q[6]) {
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    q[k] = (slots + k * FS + wave * 128)[j];
    q[3 + k] = (slots + k * FS + wave * 128 + 64)[j];
  }
}
// Its share of the face update: the + side through this face's links (the hop lands on
// l = 3, position p3), the - side as it is (l = 0).
__device__ __forceinline__ void face_stage(const f4v q[6], int wave, f4v* lh, int p3, int p0, const Cx<float> u[9]) {
  Cx<float> a[6], h[6];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    lh[(wave * 3 + k) * VB + p0] = q[3 + k];
    a[2 * k] = {q[k].x, q[k].y};
    a[2 * k + 1] = {q[k].z, q[k].w};
  }
  link_mult<float, +1>(u, a, h);
  store_half(lh, wave, p3, h);
}

}  // namespace sap4
}  // namespace qws
