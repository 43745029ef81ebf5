// sap.h -- fused SAP half-sweep kernel (one workgroup per block of one colour).
#pragma once

#include "kernels.h"

namespace qws {


enum SapFlags {
  SAP_EPI_SUPDATE = 0,   // s_c = s_c + in_c - x + kappa T^-1 H_in x ; q_c = x
  SAP_EPI_OUT = 1,       // out_c = x - kappa T^-1 H_in x            ; q_c = x
  SAP_EPI_OUT_FACE = 2,  // out_c = -kappa T^-1 H_face q + x - kappa T^-1 H_in x ; q_c = x
  SAP_EPI_NONE = 3,      // q_c = x only
  SAP_EPI_MASK = 3,
  SAP_FACE_PRO = 4,      // prologue: s_c += kappa T^-1 H_face qface
  SAP_SRC_IN = 8,        // take s_c from `in` (first sweep: s = in)
  SAP_FACE_OUT = 16,     // also write the face buffer (FP32 slots) for the next launch's prologue
  SAP_FACE_FB = 32,      // the prologue reads the face buffer instead of gathering qface
  SAP_SRC_PUPD = 64,     // with SAP_SRC_IN (FP32): first in_c = r_c + beta (in_c - omega q_c), stored
};

// The BiCGStab direction update folded into the first sweep (SAP_SRC_PUPD): `in` is
// the direction p itself, updated in place from r, q and the RHS's omega, beta.
struct SapSrcUpdate {
  float* p = nullptr;
  const float* r = nullptr;
  const float* q = nullptr;
  const Scalars* sc = nullptr;
};

// One lattice's share of a launch fused over several lattices: what a single launch
// takes as arguments, per lattice.  For the face-term kernel, kappa holds its factor.
template <typename S> struct SapPart {
  Geo g;
  const int* active;
  long long stride;
  int nrhs;
  float kappa;
  S* s;
  const S* in;
  const S* qface;
  S* qout;
  S* out;
  const S* U;
  const S* C;
  float* fb;
  long long fbs;
  SapSrcUpdate upd;
};
// A launch fused over several lattices: workgroup w runs block table[w].y of part
// table[w].x (device arrays).  The parts share the block volume (and whether the blocks
// are 4^4), the link storage, the flags and nm; xcd: map the workgroups to the table XCD by XCD.
template <typename S> struct SapMulti {
  const SapPart<S>* parts = nullptr;
  const int2* table = nullptr;
  int n = 0;
  int xcd = 1;
  int b4 = 0;        // 1: every part has 4^4 blocks (sap4.hip), 0: none has
  int rhs = 1;       // grid.y: sap_rhs_groups of the parts' largest nrhs
                     // (no padding: launch records are compared by their bytes)
};

// Over how many workgroups the nrhs right-hand sides of a block are spread: a workgroup
// takes its block's right-hand sides in turn with the links and the clover inverse held,
// so that a launch on few blocks left most of `slots` (workgroups that run at once) empty.
// The number with the shortest rounds, in units of one right-hand side; loading the
// fields is a quarter of one.  12 right-hand sides on 256 blocks (16^3 x 32, nm 6): 313 us with
// one workgroup per block, 192 with two.
inline int sap_rhs_groups(int blocks, int nrhs, int slots) {
  int best = 1;
  double time = 1e30;
  for (int k = 1; k <= nrhs; ++k) {
    const double t = (((long long)blocks * k + slots - 1) / slots) * ((nrhs + k - 1) / k + 0.25);
    if (t < 0.99 * time) time = t, best = k;
  }
  return best;
}

// Workgroups of a half-sweep launch that run at once: two per CU where the LDS holds two
// (18-real FP32 links of 256 sites take 98 KB in the general kernel: solves of 3 right-hand
// sides on 16^3 x 32 in 8x4x4x2 blocks with 512 / 256 here 21.3 / 19.9 ms, of 12 70.5 / 69.2).
inline int sap_slots(int vb, int nl, bool fp32, bool b4) { return vb == 256 && (b4 || !fp32 || nl == 12) ? 512 : 256; }

bool sap_fusable(const Geo& g);
// 4^4 blocks: the kernels of sap4.hip and sap4h.hip
bool sap_is_4444(const Geo& g);
// floats per RHS of the face buffer, or 0 when the block shape does not allow it
// (its slots must fit the iterate's LDS: 2 sum_mu Vb / B_mu <= 2 Vb)
long long sap_face_buffer_floats(const Geo& g);
// out += gamma T^-1 H_face q on the blocks of `sel` (FP32), H_face q from the face
// buffer that the preceding SAP launch of the other colour wrote (SAP_FACE_OUT)
void launch_sap_face(const Geo& g, BlockSel sel, const Batch& B, int nl, float gamma, float* out, const float* fb,
                     long long fbs, const float* U, const float* C, hipStream_t st);
template <typename S>
void launch_sap_block(const Geo& g, BlockSel sel, const Batch& B, int nl, float kappa, int nm, int flags, S* s,
                      const S* in, const S* qface, S* qout, S* out, const S* U, const S* C, float* fb,
                      long long fbs, hipStream_t st, const SapSrcUpdate& upd = SapSrcUpdate());
// The same over several lattices in one launch (FP32 storage): vb = their sites per
// block, nl their FP32 link storage; every part has a face buffer when `flags` use one.
void launch_sap_multi(const SapMulti<float>& m, int vb, int nl, int nm, int flags, hipStream_t st);
// launch_sap_block<float> and launch_sap_multi on 4^4 blocks (sap4.hip)
void launch_sap_4444(const Geo& g, BlockSel sel, const Batch& B, int nl, float kappa, int nm, int flags, float* s,
                     const float* in, const float* qface, float* qout, float* out, const float* U, const float* C,
                     float* fb, long long fbs, hipStream_t st, const SapSrcUpdate& upd);
void launch_sap_4444_multi(const SapMulti<float>& m, int nl, int nm, int flags, hipStream_t st);
// launch_sap_block<__half> on 4^4 blocks (sap4h.hip)
void launch_sap_4444_h(const Geo& g, BlockSel sel, const Batch& B, int nl, float kappa, int nm, int flags, __half* s,
                       const __half* in, const __half* qface, __half* qout, __half* out, const __half* U, const __half* C,
                       float* fb, long long fbs, hipStream_t st);
// launch_sap_face over several lattices (part.out, .fb, .fbs, .U, .C; factor in .kappa)
void launch_sap_face_multi(const SapMulti<float>& m, int vb, int nl, hipStream_t st);

}  // namespace qws
