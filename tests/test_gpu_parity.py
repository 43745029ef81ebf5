"""GPU parity: the HIP library (through its C ABI) against the CPU oracle and the
reference's golden outputs.

Tolerances (stated by the task): operator applications within 1e-13 relative in
FP64 and 1e-6 relative in FP32; composite FP32 operators (Jacobi, SAP) within a
few 1e-6; solves reach the reference's golden solution norms under check.sh
tolerances.
"""
import ctypes

import numpy as np
import pytest

import qws_amd as Q
from oracle import oracle as O
from oracle import ref_worker as RW
from tests import casekit as K

pytestmark = pytest.mark.gpu

TOL64 = 1e-13
TOL32 = 1e-6


def rel(a, b):
    return float(np.linalg.norm((np.asarray(a) - np.asarray(b)).ravel()) / np.linalg.norm(np.asarray(b).ravel()))


def random_su3(n, rng):
    """n random SU(3) matrices as QWS link arrays (n,3,3,2)."""
    z = rng.standard_normal((n, 3, 3)) + 1j * rng.standard_normal((n, 3, 3))
    q, r = np.linalg.qr(z)
    d = np.diagonal(r, axis1=1, axis2=2)
    q = q * (d / np.abs(d))[:, None, :]
    det = np.linalg.det(q)
    q[:, :, 0] /= det[:, None]  # det(q) = 1 after scaling one column by 1/det (|det| = 1)
    return np.stack([q.real, q.imag], axis=-1)


class Problem:
    def __init__(self, L, B, kappa=0.12, seed=5, su3=False, case=None):
        self.L, self.B = L, B
        V = int(np.prod(L))
        rng = np.random.default_rng(seed)
        if case is not None:
            nloc, npe, L2, B2 = K.case_geometry(case)
            assert L2 == L and B2 == B
            _, U, C, b, x0 = O.case_inputs(nloc, npe)
            self.b, self.x0 = b, x0
        else:
            U, C = K.random_su3_like(V, rng)
            if su3:
                U = random_su3(4 * V, rng).reshape(4, V, 3, 3, 2)
            self.b = rng.standard_normal((V, 3, 4, 2))
            self.x0 = rng.standard_normal((V, 3, 4, 2))
        self.U, self.C, self.kappa = U, C, kappa
        self.orc = O.Oracle(L, B, -1, kappa, U, C)
        self.lat = Q.Lattice(L, B, -1, 12 if su3 else 18, kappa=kappa)
        self.lat.load_gauge(U)
        self.lat.load_clover(C)


GEOMS = [
    ("case0", [32, 6, 4, 3], [16, 6, 4, 3]),       # QWS single rank: improper colouring
    ("proper", [8, 4, 4, 8], [2, 2, 2, 2]),        # every direction split: proper colouring
    ("mixed", [8, 4, 2, 4], [4, 2, 2, 4]),         # z, t single block: improper
    ("b4", [16, 8, 8, 8], [4, 4, 4, 4]),           # 4^4 blocks (the solver's GPU shape)
]


@pytest.fixture(scope="module", params=GEOMS, ids=[g[0] for g in GEOMS])
def prob(request):
    _, L, B = request.param
    return Problem(L, B)


@pytest.mark.parametrize("hops", [Q.HOPS_ALL, Q.HOPS_INSIDE, Q.HOPS_FACE])
@pytest.mark.parametrize("colour", [-1, 0, 1])
def test_dslash_fp64_fp32(prob, hops, colour):
    p, lat = prob, prob.lat
    for prec, dt, tol in ((Q.F64, np.float64, TOL64), (Q.F32, np.float32, TOL32)):
        src = p.b.astype(dt)
        inp = lat.spinor(prec, src)
        out = lat.spinor(prec, np.zeros_like(p.b))
        lat.dslash(out, inp, hops, colour)
        want = p.orc.dslash(src, hops, colour, out=np.zeros_like(src))
        assert rel(out.download(), want) < tol, (prec, hops, colour)


@pytest.mark.parametrize("su3", [True, False])
def test_dslash_kernel_variants(su3):
    """The FP32 full-operator kernels on 256-site blocks (global gathers, LDS-staged
    for 3 or 4 waves), in either block order, agree with the oracle and with each other
    bit for bit (same hop order and arithmetic); the autotuner keeps one pair."""
    p = Problem([16, 8, 8, 8], [4, 4, 4, 4], kappa=0.125, seed=12, su3=su3)
    src = p.b.astype(np.float32)
    inp = p.lat.spinor(Q.F32, src)
    want = p.orc.dslash(src, Q.HOPS_ALL, -1, out=np.zeros_like(src))
    outs = {}
    for order in (0, 1):  # index order, or t-z pencils inside each XCD's range
        p.lat.set_dslash_order(order)
        for k in (0, 3, 4):
            p.lat.set_dslash_kernel(k)
            out = p.lat.spinor(Q.F32, np.zeros_like(p.b))
            p.lat.dslash(out, inp, Q.HOPS_ALL, -1)
            outs[order, k] = out.download()
            assert rel(outs[order, k], want) < TOL32, (order, k)
    assert all(np.array_equal(outs[0, 0], v) for v in outs.values())
    # the FP64 operator in pencil order as well
    p.lat.set_dslash_order(1)
    o64 = p.lat.spinor(Q.F64)
    p.lat.dslash(o64, p.lat.spinor(Q.F64, p.b), Q.HOPS_ALL, -1)
    assert rel(o64.download(), p.orc.dslash(p.b, Q.HOPS_ALL, -1, out=np.zeros_like(p.b))) < TOL64
    assert p.lat.autotune_dslash(3) in (0, 3, 4) and p.lat.dslash_order() in (0, 1)
    with pytest.raises(Q.QwsError):
        p.lat.set_dslash_kernel(7)
    with pytest.raises(Q.QwsError):
        p.lat.set_dslash_order(2)
    p.lat.set_dslash_order(0)


def test_named_dslash_kernels_run_on_few_sites(monkeypatch):
    """A kernel that is named runs also where four waves per 64 sites are the automatic
    choice, which takes less than half its time there (8^4: FP32 12.2 and 5.5 us, FP64 15.3
    and 6.4); the autotuner keeps a choice that is as fast as the automatic one."""
    def lattice():
        lat = Q.Lattice([8, 8, 8, 8], [4, 4, 4, 4], -1, 12, kappa=0.125)
        lat.generate_gauge(0.3, 5)
        lat.compute_clover(1.0)
        return lat

    def us(lat, prec):
        lat.time_dslash(prec, 200)
        return min(lat.time_dslash(prec, 500) for _ in range(5)) * 1e3

    lat = lattice()
    t32, t64 = us(lat, Q.F32), us(lat, Q.F64)
    for k in (0, 3, 4):
        lat.set_dslash_kernel(k)
        assert us(lat, Q.F32) > 1.2 * t32, k
    lat.autotune_dslash(200)
    assert us(lat, Q.F32) < 1.4 * t32
    for k in ("0", "2", "3"):
        monkeypatch.setenv("QWS_MI355X_DSLASH_D", k)
        assert us(lattice(), Q.F64) > 1.2 * t64, k
    monkeypatch.delenv("QWS_MI355X_DSLASH_D")
    monkeypatch.setenv("QWS_MI355X_DSLASH", "0")
    assert us(lattice(), Q.F32) > 1.2 * t32


@pytest.mark.parametrize("L,B,su3", [([6, 3, 5, 7], [3, 3, 5, 7], False), ([4, 8, 4, 4], [2, 8, 2, 4], True),
                                     ([32, 10, 9, 23], [16, 10, 9, 23], False), ([16, 16, 32, 40], [4, 4, 4, 4], True)])
def test_operators_around_the_split_rule(L, B, su3):
    """The operators with four waves per 64 sites and the ones with a thread per site, on
    either side of the sizes where one takes over: blocks with a ragged last group of 64
    sites (105, 64, 33120 sites), whole operators of 1036 groups next to their halves of
    518, and 5120 groups of 4^4 blocks, where every staged kernel is the general one's
    equal bit for bit.  D against the oracle, and D = D_in + D_face on each colour."""
    p = Problem(L, B, kappa=0.125, seed=14, su3=su3)
    for prec, dt, tol in ((Q.F64, np.float64, TOL64), (Q.F32, np.float32, TOL32)):
        src = p.b.astype(dt)
        inp = p.lat.spinor(prec, src)
        want = p.orc.dslash(src, Q.HOPS_ALL, -1, out=np.zeros_like(src))
        outs = []
        for k in ((0, 3, 4) if prec == Q.F32 and B == [4, 4, 4, 4] else (None,)):
            if k is not None:
                p.lat.set_dslash_kernel(k)
            out = p.lat.spinor(prec)
            p.lat.dslash(out, inp, Q.HOPS_ALL, -1)
            outs.append(out.download())
        assert rel(outs[0], want) < tol
        assert all(np.array_equal(outs[0], o) for o in outs)
        out = p.lat.spinor(prec)
        for c in (0, 1):
            p.lat.dslash(out, inp, Q.HOPS_INSIDE, c)
        for c in (0, 1):
            p.lat.face(out, inp, -0.125, c)
        assert rel(out.download(), want) < tol


@pytest.mark.parametrize("L,B", [([6, 3, 5, 7], [3, 3, 5, 7]), ([4, 8, 4, 4], [2, 8, 2, 4]),
                                 ([36, 13, 15, 20], [18, 13, 15, 20])])
@pytest.mark.parametrize("nsap,nm", [(0, 3), (1, 1), (2, 2)])
def test_sap_by_steps_with_own_neighbours(L, B, nsap, nm):
    """SAP on blocks that are their own neighbours in y, z or t, whose unsolved half
    counts as zero: in one launch per pair of updates, and (2194 groups of 64 sites) in
    two; out may be the input."""
    p = Problem(L, B, kappa=0.125, seed=15)
    bs = p.b.astype(np.float32)
    x = p.lat.spinor(Q.F32, bs)
    p.lat.prec_s(x, x, nsap, nm)
    assert rel(x.download(), p.orc.prec_s(bs, nsap, nm)) < 5e-6
    x = p.lat.spinor(Q.F32, bs)
    p.lat.prec_ddd(x, x, nsap, nm)
    assert rel(x.download(), p.orc.prec_ddd_s(bs, nsap, nm)) < 5e-6


@pytest.mark.parametrize("colour", [-1, 0, 1])
def test_face_accumulate(prob, colour):
    p, lat = prob, prob.lat
    for prec, dt, tol in ((Q.F64, np.float64, TOL64), (Q.F32, np.float32, TOL32)):
        base = (0.5 * p.x0).astype(dt)
        out = lat.spinor(prec, base)
        inp = lat.spinor(prec, p.b.astype(dt))
        lat.face(out, inp, 0.37, colour)
        want = p.orc.face(base.copy(), p.b.astype(dt), 0.37, colour)
        assert rel(out.download(), want) < tol


def test_clover(prob):
    p, lat = prob, prob.lat
    out = lat.spinor(Q.F64)
    lat.clover(out, lat.spinor(Q.F64, p.b))
    assert rel(out.download(), p.orc.clover(p.b)) < TOL64


@pytest.mark.parametrize("nm", [1, 2, 3])
def test_jinv(prob, nm):
    p, lat = prob, prob.lat
    bs = p.b.astype(np.float32)
    for col in (0, 1):
        x = lat.spinor(Q.F32, np.zeros_like(p.b))
        lat.jinv(x, lat.spinor(Q.F32, bs), col, nm)
        want = p.orc.jinv_s(bs, col, nm, x=np.zeros_like(bs))
        assert rel(x.download(), want) < 3e-6


@pytest.mark.parametrize("nsap,nm", [(4, 2), (2, 3), (1, 1)])
def test_prec_ddd_and_prec_s(prob, nsap, nm):
    p, lat = prob, prob.lat
    bs = p.b.astype(np.float32)
    inp = lat.spinor(Q.F32, bs)
    out = lat.spinor(Q.F32)
    lat.prec_ddd(out, inp, nsap, nm)
    assert rel(out.download(), p.orc.prec_ddd_s(bs, nsap, nm)) < 5e-6
    lat.prec_s(out, inp, nsap, nm)
    assert rel(out.download(), p.orc.prec_s(bs, nsap, nm)) < 5e-6


@pytest.mark.parametrize("L,B,su3", [([16, 8, 8, 16], [4, 4, 4, 4], False), ([16, 8, 8, 8], [8, 4, 4, 2], False),
                                     ([16, 8, 8, 8], [8, 4, 4, 4], True)])
@pytest.mark.parametrize("nsap,nm", [(4, 2), (1, 3), (0, 2)])
def test_fused_sap_matches_unfused_and_oracle(L, B, su3, nsap, nm):
    """The fused half-sweep kernel (256- and 512-site blocks, proper colouring; the
    512-site FP32 kernel needs 12-real links) gives the same prec_ddd_s_/prec_s_ as the
    step-by-step kernels and the oracle."""
    p = Problem(L, B, kappa=0.125, seed=8, su3=su3)
    bs = p.b.astype(np.float32)
    inp = p.lat.spinor(Q.F32, bs)
    res = {}
    for fused in (True, False):
        p.lat.set_sap_fused(fused)
        o1, o2 = p.lat.spinor(Q.F32), p.lat.spinor(Q.F32)
        p.lat.prec_ddd(o1, inp, nsap, nm)
        p.lat.prec_s(o2, inp, nsap, nm)
        res[fused] = (o1.download(), o2.download())
    p.lat.set_sap_fused(True)
    want_ddd, want_s = p.orc.prec_ddd_s(bs, nsap, nm), p.orc.prec_s(bs, nsap, nm)
    for k in (True, False):
        assert rel(res[k][0], want_ddd) < 5e-6
        assert rel(res[k][1], want_s) < 5e-6
    assert rel(res[True][0], res[False][0]) < 5e-6


@pytest.mark.parametrize("L,B,su3", [([16, 8, 8, 16], [4, 4, 4, 4], True), ([16, 8, 8, 16], [4, 4, 4, 4], False),
                                     ([16, 8, 8, 8], [8, 4, 4, 4], True)])
@pytest.mark.parametrize("nsap,nm", [(2, 3), (0, 2)])
def test_fused_sap_face_buffer_is_bitwise_the_gather(L, B, su3, nsap, nm):
    """The fused SAP's face updates through the face buffer (projected, and for
    backward hops link-multiplied, face spinors written by the previous half-sweep)
    give the gathered face updates bit for bit, for one RHS and for a batch."""
    p = Problem(L, B, kappa=0.125, seed=9, su3=su3)
    rng = np.random.default_rng(5)
    srcs = [p.b.astype(np.float32), rng.standard_normal(p.b.shape).astype(np.float32)]
    res = {}
    for fb in (True, False):
        p.lat.set_sap_face_buffer(fb)
        outs = []
        for src in srcs:
            o1, o2 = p.lat.spinor(Q.F32), p.lat.spinor(Q.F32)
            p.lat.prec_ddd(o1, p.lat.spinor(Q.F32, src), nsap, nm)
            p.lat.prec_s(o2, p.lat.spinor(Q.F32, src), nsap, nm)
            outs += [o1.download(), o2.download()]
        res[fb] = outs
    p.lat.set_sap_face_buffer(True)
    for a, b in zip(res[True], res[False]):
        assert np.array_equal(a, b)
    assert rel(res[True][0], p.orc.prec_ddd_s(srcs[0], nsap, nm)) < 5e-6


@pytest.mark.parametrize("su3", [True, False])
@pytest.mark.parametrize("L,nsap,nm", [([8, 8, 8, 8], 1, 1), ([8, 8, 8, 8], 3, 2), ([24, 8, 16, 8], 2, 1),
                                       ([24, 8, 16, 8], 0, 5), ([24, 8, 16, 16], 2, 2), ([32, 16, 32, 32], 1, 2)])
def test_fused_sap_4444(L, nsap, nm, su3):
    """The FP32 kernel for 4^4 blocks (hops by link, not by site) where both neighbours
    of a block are the same one, at extents that differ in every direction, with one Jacobi
    step, with 12- and 18-real links, by eight waves a block (to 64 blocks per colour, here
    8 and 48) and by four (96), and on 1024 blocks per colour (second workgroups
    start late): the oracle's result, by the face buffer bit for bit as by gathers.  On the
    largest lattice against the step-by-step kernels.  FP32 rounding: 1e-6 at most over
    the few hundred operations behind a component, 5e-6 allowed as in the tests above."""
    big = np.prod(L) > 100000
    if big:
        lat = Q.Lattice(L, [4, 4, 4, 4], -1, 12 if su3 else 18, kappa=0.125)
        lat.generate_gauge(0.3, 1)
        lat.compute_clover(1.0)
        bs = np.random.default_rng(11).standard_normal((lat.V, 3, 4, 2)).astype(np.float32)
    else:
        p = Problem(L, [4, 4, 4, 4], kappa=0.125, seed=10, su3=su3)
        lat, bs = p.lat, p.b.astype(np.float32)
    inp = lat.spinor(Q.F32, bs)

    def both():
        o1, o2 = lat.spinor(Q.F32), lat.spinor(Q.F32)
        lat.prec_ddd(o1, inp, nsap, nm)
        lat.prec_s(o2, inp, nsap, nm)
        return o1.download(), o2.download()

    got = both()
    lat.set_sap_face_buffer(False)
    for a, b in zip(got, both()):
        assert np.array_equal(a, b)
    lat.set_sap_face_buffer(True)
    if big:
        lat.set_sap_fused(False)
        want = both()
    else:
        want = p.orc.prec_ddd_s(bs, nsap, nm), p.orc.prec_s(bs, nsap, nm)
    for a, b in zip(got, want):
        assert rel(a, b) < 5e-6


@pytest.mark.skipif(not RW.available(), reason="oracle/_ref/libqws_ref.so not built")
def test_dropin_plain_dd_solvers_and_helpers_case0():
    """bicgstab_dd_s_/bicgstab_dd_d_ (plain BiCGStab on D) through the QWS ABI on
    data/CASE0's fields agree with the reference's own (oracle/_ref) from the same initial
    guess: same stopping rule (1e-6 FP32, 1e-14 FP64), iteration counts within 5% (the
    reference reduces in FP32 for FP32, this library in FP64), solutions to the
    tolerance's accuracy; ddd_eo_s_ of both domains reproduces data/CASE0's ddd_s_ norm;
    the plain reorders are exact casts."""
    L = Q.lib()
    nloc = [32, 6, 4, 3]
    _, U, C, b, x0 = O.case_inputs(nloc)
    ci = lambda v: ctypes.byref(ctypes.c_int(v))
    keep = [(ctypes.c_int * 4)(1, 1, 1, 1), (ctypes.c_int * 4)(1, 1, 1, -1), ctypes.c_int(0), ctypes.c_int(1),
            (ctypes.c_int * 4)(1, 2, 2, 2)]
    L.qws_init_(ci(32), ci(6), ci(4), ci(3), keep[0], keep[1], ctypes.byref(keep[2]), ctypes.byref(keep[3]), keep[4])
    vold = ctypes.c_int.in_dll(L, "vold").value
    vols = ctypes.c_int.in_dll(L, "vols").value

    def glob(name, ct, n):
        return np.ctypeslib.as_array((ct * n).from_address(ctypes.c_void_p.in_dll(L, name).value))

    glob("glud", ctypes.c_double, vold * 8 * 144)[:] = RW.links_to_aosoa(U, nloc, 8).ravel()
    glob("glus", ctypes.c_float, vols * 8 * 288)[:] = RW.links_to_aosoa(U.astype(np.float32), nloc, 16).ravel()
    glob("clvd", ctypes.c_double, vold * 2 * 576)[:] = RW.clover_to_aosoa(C, nloc, 8).ravel()
    glob("clvs", ctypes.c_float, vols * 2 * 1152)[:] = RW.clover_to_aosoa(C.astype(np.float32), nloc, 16).ravel()
    ctypes.c_double.in_dll(L, "kappa").value = 0.05
    ctypes.c_double.in_dll(L, "mkappa").value = -0.05
    ctypes.c_double.in_dll(L, "kappa2").value = 0.0025
    L.qws_mi355x_fields_modified_()
    bd = RW.spinor_to_aosoa(b, nloc, 8)
    bs = RW.spinor_to_aosoa(b.astype(np.float32), nloc, 16)
    itd, its = ctypes.c_int(0), ctypes.c_int(0)
    xd = RW.spinor_to_aosoa(x0, nloc, 8)
    L.bicgstab_dd_d_(_ptr(xd), _ptr(bd), ctypes.byref(itd), ci(1000))
    xs = RW.spinor_to_aosoa(x0.astype(np.float32), nloc, 16)
    L.bicgstab_dd_s_(_ptr(xs), _ptr(bs), ctypes.byref(its), ci(1000))
    rd, rs = np.zeros_like(bd), np.zeros_like(bs)
    L.ddd_d_(_ptr(rd), _ptr(xd))
    L.ddd_s_(_ptr(rs), _ptr(xs))
    # ddd_eo_s_ on both domains (qws.cc:641-644) is ddd_s_
    eo = np.zeros_like(bs)
    for d in (0, 1):
        L.ddd_eo_s_(_ptr(eo), _ptr(bs), ci(d))
    full = np.zeros_like(bs)
    L.ddd_s_(_ptr(full), _ptr(bs))
    # plain reorders: exact casts between the two host layouts
    s32 = np.zeros_like(bs)
    L.fermi_reorder_d2s_dd_(_ptr(s32), _ptr(bd))
    d64 = np.zeros_like(bd)
    L.fermi_reorder_s2d_dd_(_ptr(d64), _ptr(s32))
    L.qws_finalize_()
    # (the reference defines ddd_s_ this way, so its golden norm applies; this library's
    # ddd_s_ is one fused operator, equal to rounding)
    assert K.check_value("ddd_s_", O.norm2(eo), K.expected("CASE0", "ddd_s_"))
    assert rel(eo, full) < 1e-6
    assert np.array_equal(s32, bs)
    assert np.array_equal(RW.spinor_from_aosoa(d64, nloc, 8), b.astype(np.float32).astype(np.float64))
    assert 2 < itd.value < 1000 and 2 < its.value < 1000
    assert O.norm2(bd - rd) < 1e-25 * O.norm2(bd)
    assert O.norm2(bs - rs) < 1e-10 * O.norm2(bs)
    ref = RW.call(nloc, 0.05, U, C, b, ["bicgstab_dd_d", "bicgstab_dd_s"], x0=x0, maxiter=1000)
    # ~200 (FP64) and ~90 (FP32) iterations: the differently ordered sums may move the
    # stopping iteration by a few
    for it, name in ((itd.value, "bicgstab_dd_d_iter"), (its.value, "bicgstab_dd_s_iter")):
        assert abs(int(ref[name]) - it) <= max(2, 0.05 * int(ref[name])), (name, it, int(ref[name]))
    assert rel(RW.spinor_from_aosoa(xd, nloc, 8), ref["bicgstab_dd_d"]) < 1e-12
    assert rel(RW.spinor_from_aosoa(xs, nloc, 16), ref["bicgstab_dd_s"]) < 1e-5


def _case0_dropin(L):
    """qws_init_ on data/CASE0's geometry with its fields in the host arrays (kappa 0.05)."""
    nloc = [32, 6, 4, 3]
    _, U, C, b, x0 = O.case_inputs(nloc)
    ci = lambda v: ctypes.byref(ctypes.c_int(v))
    keep = [(ctypes.c_int * 4)(1, 1, 1, 1), (ctypes.c_int * 4)(1, 1, 1, -1), ctypes.c_int(0), ctypes.c_int(1),
            (ctypes.c_int * 4)(1, 2, 2, 2)]
    L.qws_init_(ci(32), ci(6), ci(4), ci(3), keep[0], keep[1], ctypes.byref(keep[2]), ctypes.byref(keep[3]), keep[4])
    vold = ctypes.c_int.in_dll(L, "vold").value
    vols = ctypes.c_int.in_dll(L, "vols").value

    def glob(name, ct, n):
        return np.ctypeslib.as_array((ct * n).from_address(ctypes.c_void_p.in_dll(L, name).value))

    glob("glud", ctypes.c_double, vold * 8 * 144)[:] = RW.links_to_aosoa(U, nloc, 8).ravel()
    glob("glus", ctypes.c_float, vols * 8 * 288)[:] = RW.links_to_aosoa(U.astype(np.float32), nloc, 16).ravel()
    glob("clvd", ctypes.c_double, vold * 2 * 576)[:] = RW.clover_to_aosoa(C, nloc, 8).ravel()
    glob("clvs", ctypes.c_float, vols * 2 * 1152)[:] = RW.clover_to_aosoa(C.astype(np.float32), nloc, 16).ravel()
    ctypes.c_double.in_dll(L, "kappa").value = 0.05
    ctypes.c_double.in_dll(L, "mkappa").value = -0.05
    ctypes.c_double.in_dll(L, "kappa2").value = 0.0025
    L.qws_mi355x_fields_modified_()
    return nloc, U, C, b, x0, keep, vold, vols


@pytest.mark.skipif(not RW.available(), reason="oracle/_ref/libqws_ref.so not built")
def test_dropin_remaining_entry_points_case0(capfd):
    """The QWS entry points not covered elsewhere, on data/CASE0's host arrays: the FP64
    domain-local and face terms and the clover multiplies reproduce CASE0's golden norms
    (main.cc:636-690); jinv_ddd_in_s_, prec_ddd_s_, prec_s_ and bicgstab_precdd_s_ agree
    with the reference library (oracle/_ref) on the same input; the renormalising
    reorders follow their closed forms (out = in / |in|, out = in * dnorm);
    check_residual_s_ prints |b - prec_ddd_s_(x)| / sqrt(bnorm); and a solve with SAP
    blocks set by qws_mi355x_set_sap_blocks_ still meets its tolerance."""
    L = Q.lib()
    nloc, U, C, b, x0, keep, vold, vols = _case0_dropin(L)
    ci = lambda v: ctypes.byref(ctypes.c_int(v))
    cd = lambda v: ctypes.byref(ctypes.c_double(v))
    bd = RW.spinor_to_aosoa(b, nloc, 8)
    bs = RW.spinor_to_aosoa(b.astype(np.float32), nloc, 16)
    got = {}
    out = np.zeros_like(bd)
    L.ddd_out_pre_d_(_ptr(bd), ci(0))
    L.ddd_out_pos_d_(_ptr(out), _ptr(bd), ci(0))
    got["ddd_out_pre|pos_d_"] = O.norm2(out)
    out[:] = 0
    L.ddd_in_d_(_ptr(out), _ptr(bd), ci(0))
    got["ddd_in_d_"] = O.norm2(out)
    inp = np.ascontiguousarray(bd.reshape(2 * vold, -1)[:vold])
    o1 = inp.copy()
    L.clvd_vm_(ci(0), _ptr(o1))
    got["clvd_vm_"] = O.norm2(o1)
    o2 = np.zeros_like(inp)
    L.clvd_vm2_(ci(0), _ptr(o2), _ptr(inp))
    got["clvd_vm2_"] = O.norm2(o2)
    # the SAP pieces and the inner solver (nsap 4, nm 2; 6 fixed inner iterations)
    mine = {}
    for d in (0, 1):
        o = np.zeros_like(bs)
        L.jinv_ddd_in_s_(_ptr(o[d]), _ptr(bs[d]), ci(d), ci(2))
        mine[f"jinv{d}"] = o
    o = np.zeros_like(bs)
    L.prec_ddd_s_(_ptr(o), _ptr(bs), ci(4), ci(2))
    mine["prec_ddd_s"] = o
    o = np.zeros_like(bs)
    L.prec_s_(_ptr(o), _ptr(bs), ci(4), ci(2))
    mine["prec_s"] = o
    o = np.zeros_like(bs)
    it = ctypes.c_int(0)
    L.bicgstab_precdd_s_(_ptr(o), _ptr(bs), cd(-1.0), ctypes.byref(it), ci(6), ci(4), ci(2))
    mine["bicgstab_precdd_s"] = o
    # renormalising reorders (reordering.cc:108-204)
    L.fermi_reorder_d2s_dd_renorm_.argtypes = [ctypes.c_void_p] * 3
    L.fermi_reorder_s2d_dd_renorm_.argtypes = [ctypes.c_void_p] * 3
    dn = ctypes.c_double(0)
    s32 = np.zeros_like(bs)
    L.fermi_reorder_d2s_dd_renorm_(_ptr(s32), _ptr(bd), ctypes.byref(dn))
    back = np.zeros_like(bd)
    L.fermi_reorder_s2d_dd_renorm_(_ptr(back), _ptr(s32), ctypes.byref(dn))
    # check_residual_s_ of the inner solution
    L.check_residual_s_.argtypes = [ctypes.c_void_p] * 6
    bn = ctypes.c_float(np.float32(O.norm2(bs)))
    capfd.readouterr()
    L.check_residual_s_(_ptr(mine["bicgstab_precdd_s"]), _ptr(bs), ci(6), ctypes.byref(bn), ci(4), ci(2))
    printed = capfd.readouterr().out
    w = np.zeros_like(bs)
    L.prec_ddd_s_(_ptr(w), _ptr(mine["bicgstab_precdd_s"]), ci(4), ci(2))
    # SAP blocks of 8x6x4x3 instead of the two x-halves
    L.qws_mi355x_set_sap_blocks_((ctypes.c_int * 4)(8, 6, 4, 3))
    x = RW.spinor_to_aosoa(x0, nloc, 8)
    L.bicgstab_dd_mix_(_ptr(x), _ptr(bd), cd(1e-12), ctypes.byref(it), ci(50), cd(1e-4), ci(50), ci(4), ci(2))
    r = np.zeros_like(bd)
    L.ddd_d_(_ptr(r), _ptr(x))
    L.qws_finalize_()
    for name, v in got.items():
        assert K.check_value(name, v, K.expected("CASE0", name)), (name, v)
    ref = RW.call(nloc, 0.05, U, C, b, ["jinv0", "jinv1", "prec_ddd_s", "prec_s", "bicgstab_precdd_s"], nsap=4,
                  nm=2, tol_s=-1.0, maxiter_s=6)
    # FP32 operators to rounding; the solver after 6 iterations also carries the
    # difference of FP32 (reference) and FP64 (this library) reductions
    for name, v in mine.items():
        tol = 2e-5 if name == "bicgstab_precdd_s" else 2e-6
        assert rel(RW.spinor_from_aosoa(v, nloc, 16), ref[name]) < tol, name
    nb = np.sqrt(O.norm2(bd))
    assert abs(dn.value - nb) < 1e-14 * nb
    s32p = RW.spinor_from_aosoa(s32, nloc, 16)
    assert rel(s32p, (b / nb).astype(np.float32)) < 1e-7
    assert np.array_equal(RW.spinor_from_aosoa(back, nloc, 8), s32p.astype(np.float64) * dn.value)
    line = [t for t in printed.splitlines() if t.startswith("@C")]
    assert len(line) == 1 and int(line[0].split()[1]) == 6, printed
    err = np.sqrt(O.norm2((bs - w).astype(np.float64)) / float(bn.value))
    assert abs(float(line[0].split()[2]) - err) < 1e-4 * err + 1e-12
    assert 1 < it.value < 50
    assert O.norm2(bd - r) < 1e-22 * O.norm2(bd)


def test_dropin_links12_matches_links18_on_su3_fields():
    """qws_mi355x_set_links12_: with SU(3) links in the host arrays, the drop-in's FP32
    operator, SAP preconditioner and mixed solve with 12-real device links (row 2
    rebuilt) agree with the 18-real ones to FP32 rounding; the solve meets 1e-10."""
    import bench
    L = Q.lib()
    nloc = [32, 8, 8, 8]
    g = Q.Lattice(nloc, [4, 4, 4, 4], -1, 12, kappa=0.13)
    g.generate_gauge(0.3, 5)
    g.compute_clover(1.0)
    U, C, b = g.gauge(), g.clover_field(), g.gaussian(Q.F64, 6).download()
    g.close()
    ci = lambda v: ctypes.byref(ctypes.c_int(v))
    cd = lambda v: ctypes.byref(ctypes.c_double(v))
    keep = [(ctypes.c_int * 4)(1, 1, 1, 1), (ctypes.c_int * 4)(1, 1, 1, -1), ctypes.c_int(0), ctypes.c_int(1),
            (ctypes.c_int * 4)(1, 2, 2, 2)]
    L.qws_init_(ci(32), ci(8), ci(8), ci(8), keep[0], keep[1], ctypes.byref(keep[2]), ctypes.byref(keep[3]), keep[4])

    def fill(name, arr):
        dst = np.ctypeslib.as_array((ctypes.c_byte * arr.nbytes).from_address(ctypes.c_void_p.in_dll(L, name).value))
        dst[:] = arr.view(np.int8).ravel()

    fill("glud", bench.qws_host_layout(U, "links", nloc, 8))
    fill("glus", bench.qws_host_layout(U.astype(np.float32), "links", nloc, 16))
    fill("clvd", bench.qws_host_layout(C, "clover", nloc, 8))
    fill("clvs", bench.qws_host_layout(C.astype(np.float32), "clover", nloc, 16))
    for name, v in (("kappa", 0.13), ("mkappa", -0.13), ("kappa2", 0.13 ** 2)):
        ctypes.c_double.in_dll(L, name).value = v
    L.qws_mi355x_fields_modified_()
    L.qws_mi355x_set_sap_blocks_((ctypes.c_int * 4)(4, 4, 4, 4))
    bd = bench.qws_host_layout(b, "spinor", nloc, 8)
    bs = bench.qws_host_layout(b.astype(np.float32), "spinor", nloc, 16)
    L.bicgstab_dd_mix_status_.restype = ctypes.c_int
    res = {}
    for on in (0, 1):
        L.qws_mi355x_set_links12_(ci(on))
        d = np.zeros_like(bs)
        L.ddd_s_(_ptr(d), _ptr(bs))
        m = np.zeros_like(bs)
        L.prec_ddd_s_(_ptr(m), _ptr(bs), ci(2), ci(6))
        x = np.zeros_like(bd)
        it, tr = ctypes.c_int(0), ctypes.c_double(0)
        rc = L.bicgstab_dd_mix_status_(_ptr(x), _ptr(bd), cd(1e-11), ctypes.byref(it), ci(40), cd(1e-3), ci(80),
                                       ci(2), ci(6), ctypes.byref(tr))
        res[on] = (d, m, x, rc, it.value, tr.value)
    L.qws_finalize_()
    a, b18 = res[1], res[0]
    assert rel(a[0], b18[0]) < 1e-6
    assert rel(a[1], b18[1]) < 1e-5
    assert a[3] == 0 and b18[3] == 0 and a[5] < 1e-10 and b18[5] < 1e-10, (a[3:], b18[3:])
    assert rel(a[2], b18[2]) < 1e-7


def test_bicgstab_direction_update_in_the_sap_sweep_is_bitwise_the_separate_pass():
    """The inner BiCGStab's direction update p = r + beta (p - omega q) done by the first
    fused SAP sweep of the next preconditioner application gives the separate update
    pass's results bit for bit: the inner solve alone (x, iterations), a mixed solve,
    and a batch of Gaussian and point sources."""
    lat = Q.Lattice([8, 8, 8, 16], [4, 4, 4, 4], -1, 12, kappa=0.13)
    lat.generate_gauge(0.3, 11)
    lat.compute_clover(1.0)
    srcs = [lat.gaussian(Q.F64, 100), lat.gaussian(Q.F64, 101), lat.point(Q.F64, (0, 0, 0, 0), 0, 0),
            lat.point(Q.F64, (3, 1, 2, 5), 2, 1)]
    b32 = lat.spinor(Q.F32, srcs[0].download().astype(np.float32))
    prm = dict(nsap=2, nm=3, tol=1e-10, maxiter=30, tol_s=1e-4, maxiter_s=50)
    res = {}
    for on in (True, False):
        lat.set_sap_source_update(on)
        x = lat.spinor(Q.F32)
        it = lat.bicgstab_precdd(x, b32, 1e-6, 80, 2, 3)
        xd = lat.spinor(Q.F64)
        st = lat.solve(xd, srcs[1], **prm)
        xs = [lat.spinor(Q.F64) for _ in srcs]
        sts = lat.solve_batch(xs, srcs, **prm)
        res[on] = (x.download(), it, xd.download(), (st["outer_iters"], st["inner_iters"]), st["true_residual"],
                   [v.download() for v in xs], [(s_["outer_iters"], s_["inner_iters"]) for s_ in sts])
    lat.set_sap_source_update(True)
    a, b = res[True], res[False]
    print("inner solve", a[1], "solve", a[3], "batch", a[6])
    assert a[1] == b[1] and 1 < a[1] < 80
    assert np.array_equal(a[0], b[0])
    assert np.array_equal(a[2], b[2]) and a[3] == b[3]
    assert 0 < a[4] < 1e-9
    assert a[6] == b[6]
    for u, v in zip(a[5], b[5]):
        assert np.array_equal(u, v)


def test_time_sap_runs_the_fused_kernel():
    """The SAP timing entry point runs the fused launches of one preconditioner
    application (FP32 and FP16 storage), leaves the operator's results unchanged and
    reports a positive device time; blocks the fused kernel cannot take are refused."""
    p = Problem([16, 8, 8, 16], [4, 4, 4, 4], kappa=0.125, seed=8, su3=True)
    bs = p.b.astype(np.float32)
    inp = p.lat.spinor(Q.F32, bs)
    o1, o2 = p.lat.spinor(Q.F32), p.lat.spinor(Q.F32)
    p.lat.prec_ddd(o1, inp, 2, 3)
    for prec in (Q.F32, Q.F16):
        ms = p.lat.time_sap(prec, 3, 2, 3)
        assert 0 < ms < 100, (prec, ms)
    p.lat.prec_ddd(o2, inp, 2, 3)
    assert np.array_equal(o1.download(), o2.download())
    q = Problem([8, 4, 4, 8], [2, 2, 2, 2])
    with pytest.raises(Q.QwsError):
        q.lat.time_sap(Q.F32, 1, 2, 2)


def test_stream_bandwidth_probe():
    """The HBM probe runs (copy and a 6:1 read-mostly sum) and reports a plausible
    rate; bad arguments are refused."""
    for nin in (1, 6):
        for one in (False, True):
            g = Q.stream_bandwidth(64 << 20, nin, 3, one_stream=one)
            assert 100 < g < 20000, (nin, one, g)
    with pytest.raises(Q.QwsError):
        Q.stream_bandwidth(1024, 1, 1)
    with pytest.raises(Q.QwsError):
        Q.stream_bandwidth(64 << 20, 17, 1, one_stream=True)


def test_inner_bicgstab(prob):
    p, lat = prob, prob.lat
    bs = (p.b / np.sqrt(O.norm2(p.b))).astype(np.float32)
    x = lat.spinor(Q.F32)
    it = lat.bicgstab_precdd(x, lat.spinor(Q.F32, bs), -1.0, 3, 4, 2)
    want, it_o = p.orc.bicgstab_precdd_s(bs, -1.0, 3, 4, 2)
    assert it == it_o == 3
    assert rel(x.download(), want) < 1e-4


def test_inner_bicgstab_stops_at_either_half_step():
    """The inner solve with a tolerance (bicgstab_precdd_s.cc:594) ends after the half-step
    whose residual meets it, the first or the second of an iteration, and x then holds that
    half-step's update: equal to the oracle at both kinds of exit (which kind each tolerance
    gives is read off the oracle: an exit after the second half-step equals the fixed-count
    run of the same iterations)."""
    p = Problem([16, 8, 8, 8], [4, 4, 4, 4])
    lat = p.lat
    bs = (p.b / np.sqrt(O.norm2(p.b))).astype(np.float32)
    halves = set()
    for tol in (1e-2, 1e-3, 1e-5):
        want, it_o = p.orc.bicgstab_precdd_s(bs, tol, 50, 4, 2)
        fixed, _ = p.orc.bicgstab_precdd_s(bs, -1.0, it_o, 4, 2)
        halves.add((it_o, 2 if np.array_equal(want, fixed) else 1))
        x = lat.spinor(Q.F32)
        it = lat.bicgstab_precdd(x, lat.spinor(Q.F32, bs), tol, 50, 4, 2)
        print(f"[inner] tol {tol:g}: {it} / {it_o} iterations", flush=True)
        assert it == it_o
        assert rel(x.download(), want) < 1e-4
    assert {h for _, h in halves} == {1, 2}, halves  # both exits exercised
    assert any(i > 1 and h == 1 for i, h in halves)  # a first-half exit after a full iteration
    lat.close()


def test_fp64_dslash_kernels_agree_bitwise(monkeypatch):
    """The FP64 full operator on 256-site blocks: the LDS-staged kernels (default, and the
    3-wave build) give the gathering kernel's result bit for bit, and match the oracle."""
    p = Problem([16, 8, 8, 8], [4, 4, 4, 4], seed=12)
    digests = []
    for kd in ("0", "2", "3"):
        monkeypatch.setenv("QWS_MI355X_DSLASH_D", kd)  # read when a lattice is created
        lat = Q.Lattice(p.L, p.B, -1, 18, kappa=p.kappa)
        lat.load_gauge(p.U)
        lat.load_clover(p.C)
        o = lat.spinor(Q.F64)
        lat.dslash(o, lat.spinor(Q.F64, p.b))
        digests.append(o.digest())
        if kd == "2":
            assert rel(o.download(), p.orc.dslash(p.b)) < TOL64
        lat.close()
    assert digests[0] == digests[1] == digests[2]


@pytest.mark.parametrize("links", [12, 18])
def test_full_operators_beyond_the_last_level_cache(monkeypatch, links):
    """24^3 x 32 in 4^4 blocks, 297 MB and more in FP32 and 679 MB in FP64: clover and results
    past the caches, blocks in chunks over the XCDs in index order and in contiguous ranges in
    pencil order.  Every kernel gives the gathering one's result bit for bit, the oracle's to
    rounding; so does D by halves of 3456 groups of 64 sites (FP64 by four waves per group)."""
    L = [24, 24, 24, 32]
    lat = Q.Lattice(L, [4, 4, 4, 4], -1, links, kappa=0.12)
    lat.generate_gauge(0.3, 7)
    lat.compute_clover(1.0)
    U, C = lat.gauge(), lat.clover_field()
    orc = O.Oracle(L, [4, 4, 4, 4], -1, 0.12, U, C)
    b = np.random.default_rng(31).standard_normal((lat.V, 3, 4, 2))
    for prec, dt, tol in ((Q.F32, np.float32, TOL32), (Q.F64, np.float64, TOL64)):
        want = orc.dslash(b.astype(dt))
        digests = set()
        for kd in (("0", "2", "3") if prec == Q.F64 else ("2",)):
            monkeypatch.setenv("QWS_MI355X_DSLASH_D", kd)
            one = Q.Lattice(L, [4, 4, 4, 4], -1, links, kappa=0.12)
            one.load_gauge(U)
            one.load_clover(C)
            inp, o = one.spinor(prec, b.astype(dt)), one.spinor(prec)
            for order in (0, 1):
                one.set_dslash_order(order)
                for k in ((0, 3, 4) if prec == Q.F32 else (None,)):
                    if k is not None:
                        one.set_dslash_kernel(k)
                    o.zero()
                    one.dslash(o, inp)
                    digests.add(o.digest())
            one.close()
        o = lat.spinor(prec)
        lat.dslash(o, lat.spinor(prec, b.astype(dt)))
        assert digests == {o.digest()}, prec
        assert rel(o.download(), want) < tol
    lat.close()
    lat = Q.Lattice(L, [12, 24, 24, 32], -1, links, kappa=0.12)
    lat.load_gauge(U)
    lat.load_clover(C)
    o = lat.spinor(Q.F64)
    lat.dslash(o, lat.spinor(Q.F64, b))
    assert rel(o.download(), want) < TOL64
    lat.close()


@pytest.mark.parametrize("B,su3", [([8, 4, 4, 2], True), ([8, 4, 4, 2], False), ([4, 4, 2, 8], True)])
def test_fused_sap_on_other_256_site_blocks(B, su3):
    """The general half-sweep kernel on blocks of 256 sites that are not 4^4, with 12-real and
    18-real links: face buffer and gathers bit for bit alike, and the oracle's result."""
    p = Problem([16, 8, 8, 16], B, kappa=0.125, seed=9, su3=su3)
    src = p.b.astype(np.float32)
    res = []
    for fb in (True, False):
        p.lat.set_sap_face_buffer(fb)
        o1, o2 = p.lat.spinor(Q.F32), p.lat.spinor(Q.F32)
        p.lat.prec_ddd(o1, p.lat.spinor(Q.F32, src), 2, 3)
        p.lat.prec_s(o2, p.lat.spinor(Q.F32, src), 2, 3)
        res.append((o1.download(), o2.download()))
    for a, b in zip(*res):
        assert np.array_equal(a, b)
    assert rel(res[0][0], p.orc.prec_ddd_s(src, 2, 3)) < 5e-6
    assert rel(res[0][1], p.orc.prec_s(src, 2, 3)) < 5e-6


def test_links12_reconstruction():
    """12-real FP32 links (third row rebuilt) equal 18-real storage for SU(3) links."""
    p = Problem([8, 8, 4, 8], [4, 4, 2, 4], su3=True, seed=11)
    lat18 = Q.Lattice(p.L, p.B, -1, 18, kappa=p.kappa)
    lat18.load_gauge(p.U)
    lat18.load_clover(p.C)
    bs = p.b.astype(np.float32)
    outs = []
    for lat in (p.lat, lat18):
        o = lat.spinor(Q.F32)
        lat.dslash(o, lat.spinor(Q.F32, bs))
        outs.append(o.download())
    assert rel(outs[0], outs[1]) < 1e-6
    assert rel(outs[0], p.orc.dslash(bs)) < TOL32


# ---------------------------------------------------------------- solves vs golden norms
@pytest.mark.parametrize("case", ["CASE0", "CASE_4111_1111", "CASE1", "CASE7"])
def test_dd_mixed_solve_golden(case):
    """bicgstab_dd_mix_ with the driver's settings (main.cc:262-312) reaches the
    reference's solution: |x|^2 at 1e-14, |b - D x|^2 < 1e-15."""
    nloc, npe, L, B = K.case_geometry(case)
    _, U, C, b, x0 = O.case_inputs(nloc, npe)
    lat = Q.Lattice(L, B, -1, 18, kappa=0.05)
    lat.load_gauge(U)
    lat.load_clover(C)
    x = lat.spinor(Q.F64, x0)
    bb = lat.spinor(Q.F64, b)
    st = lat.solve(x, bb, nsap=4, nm=2, tol=-1, maxiter=6, tol_s=-1, maxiter_s=50)
    assert st["outer_iters"] == 6 and st["inner_iters"] == 500
    xs = x.download()
    orc = O.Oracle(L, B, -1, 0.05, U, C)
    r = b - orc.dslash(xs)
    assert O.norm2(r) < 1e-15
    assert K.check_value("xnorm^2", O.norm2(xs), K.expected(case, "xnorm^2", "DD"))
    assert st["true_residual"] < 1e-10


def test_solve_to_true_residual():
    p = Problem([8, 8, 8, 8], [4, 4, 4, 4], kappa=0.1, seed=21)
    x = p.lat.spinor(Q.F64)
    st = p.lat.solve(x, p.lat.spinor(Q.F64, p.b), nsap=4, nm=2, tol=1e-11, maxiter=50, tol_s=1e-3,
                     maxiter_s=20, true_tol=1e-10, max_restarts=3)
    assert st["true_residual"] <= 1e-10
    r = p.b - p.orc.dslash(x.download())
    assert np.sqrt(O.norm2(r) / O.norm2(p.b)) <= 1e-10


# ---------------------------------------------------------------- QWS drop-in ABI
def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def test_dropin_abi_case0():
    """The QWS entry points on QWS's host layout reproduce data/CASE0."""
    L = Q.lib()
    nloc = [32, 6, 4, 3]
    _, U, C, b, x0 = O.case_inputs(nloc)
    ci = lambda v: ctypes.byref(ctypes.c_int(v))
    keep = [(ctypes.c_int * 4)(1, 1, 1, 1), (ctypes.c_int * 4)(1, 1, 1, -1), ctypes.c_int(0), ctypes.c_int(1),
            (ctypes.c_int * 4)(1, 2, 2, 2)]
    L.qws_init_(ci(32), ci(6), ci(4), ci(3), keep[0], keep[1], ctypes.byref(keep[2]), ctypes.byref(keep[3]), keep[4])
    vold = ctypes.c_int.in_dll(L, "vold").value
    vols = ctypes.c_int.in_dll(L, "vols").value

    def glob(name, ct, n):
        return np.ctypeslib.as_array((ct * n).from_address(ctypes.c_void_p.in_dll(L, name).value))

    glob("glud", ctypes.c_double, vold * 8 * 144)[:] = RW.links_to_aosoa(U, nloc, 8).ravel()
    glob("glus", ctypes.c_float, vols * 8 * 288)[:] = RW.links_to_aosoa(U.astype(np.float32), nloc, 16).ravel()
    glob("clvd", ctypes.c_double, vold * 2 * 576)[:] = RW.clover_to_aosoa(C, nloc, 8).ravel()
    glob("clvs", ctypes.c_float, vols * 2 * 1152)[:] = RW.clover_to_aosoa(C.astype(np.float32), nloc, 16).ravel()
    ctypes.c_double.in_dll(L, "kappa").value = 0.05
    ctypes.c_double.in_dll(L, "mkappa").value = -0.05
    ctypes.c_double.in_dll(L, "kappa2").value = 0.0025
    L.qws_mi355x_fields_modified_()
    bd = RW.spinor_to_aosoa(b, nloc, 8)
    bs = RW.spinor_to_aosoa(b.astype(np.float32), nloc, 16)
    out = np.zeros_like(bd)
    L.ddd_d_(_ptr(out), _ptr(bd))
    assert K.check_value("ddd_d_", O.norm2(out), K.expected("CASE0", "ddd_d_"))
    outs = np.zeros_like(bs)
    L.ddd_s_(_ptr(outs), _ptr(bs))
    assert K.check_value("ddd_s_", O.norm2(outs), K.expected("CASE0", "ddd_s_"))
    outs[:] = 0
    L.ddd_in_s_(_ptr(outs), _ptr(bs), ci(0))
    assert K.check_value("ddd_in_s_", O.norm2(outs), K.expected("CASE0", "ddd_in_s_"))
    outs[:] = 0
    L.ddd_out_pre_s_(_ptr(bs), ci(0))
    L.ddd_out_pos_s_.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_float]
    L.ddd_out_pos_s_(_ptr(outs), _ptr(bs), ci(0), ctypes.c_float(-0.05))
    assert K.check_value("ddd_out_pre|pos_s_", O.norm2(outs), K.expected("CASE0", "ddd_out_pre|pos_s_"))
    # the mixed solve (main.cc:280)
    x = RW.spinor_to_aosoa(x0, nloc, 8)
    it = ctypes.c_int(0)
    cd = lambda v: ctypes.byref(ctypes.c_double(v))
    L.bicgstab_dd_mix_(_ptr(x), _ptr(bd), cd(-1.0), ctypes.byref(it), ci(6), cd(-1.0), ci(50), ci(4), ci(2))
    assert it.value == 6
    r = np.zeros_like(bd)
    L.ddd_d_(_ptr(r), _ptr(x))
    assert O.norm2(bd - r) < 1e-15
    assert K.check_value("xnorm^2", O.norm2(x), K.expected("CASE0", "xnorm^2", "DD"))
    # the status variant: same solution bit for bit, plus the outcome and the true residual
    L.bicgstab_dd_mix_status_.restype = ctypes.c_int
    xs = RW.spinor_to_aosoa(x0, nloc, 8)
    its, tr = ctypes.c_int(0), ctypes.c_double(0)
    rc = L.bicgstab_dd_mix_status_(_ptr(xs), _ptr(bd), cd(-1.0), ctypes.byref(its), ci(6), cd(-1.0), ci(50), ci(4),
                                   ci(2), ctypes.byref(tr))
    assert rc == 0 and its.value == 6 and np.array_equal(xs, x)
    assert 0 <= tr.value < 1e-9 and abs(tr.value - np.sqrt(O.norm2(bd - r) / O.norm2(bd))) < 1e-12
    # a tolerance 2 outer iterations do not meet: 1, conviter = maxiter
    xs = RW.spinor_to_aosoa(x0, nloc, 8)
    # (inner solves to 0.1 only: two outer iterations cannot reach 1e-14)
    rc = L.bicgstab_dd_mix_status_(_ptr(xs), _ptr(bd), cd(1e-14), ctypes.byref(its), ci(2), cd(0.1), ci(50), ci(4),
                                   ci(2), ctypes.byref(tr))
    assert rc == 1 and its.value == 2 and tr.value > 1e-10, (rc, its.value, tr.value)
    rc = L.bicgstab_dd_mix_status_(_ptr(xs), _ptr(bd), cd(1e-14), ctypes.byref(its), ci(2), cd(1e-6), ci(50), ci(11),
                                   ci(2), ctypes.byref(tr))
    assert rc == -2 and tr.value == -1
    L.qws_finalize_()
    rc = L.bicgstab_dd_mix_status_(_ptr(xs), _ptr(bd), cd(1e-14), ctypes.byref(its), ci(2), cd(1e-6), ci(50), ci(4),
                                   ci(2), ctypes.byref(tr))
    assert rc == -1
