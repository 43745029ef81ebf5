"""Performance cases: the work that a user of this solver has it do, through the
device-resident interface (qws_amd, the binding of the qwsg_* entry points).

A case names an operation and its lattice:

  dslash    out = D in, the full Wilson-clover operator (FP32 or FP64)
  prec_ddd  out = D M_SAP in, the SAP-preconditioned operator of the inner solver (FP32)
  mtilde    the even/odd Schur operator on the even sites (FP32 or FP64)
  solve     D x = b from x = 0 to a 1e-10 FP64 true residual; nrhs sources in one batch,
            SAP iterates stored in FP32 or FP16
  eo_solve  mtilde x = b by the even/odd BiCGStab (FP64) from x = 0

Inputs: SU(3) links near unity (the size of exp(0.3 i H)), a Hermitian clover inverse
close to 1/2 (1/2 is the free one), Gaussian spinors.  The solves' sources are b = D y of
a Gaussian y, so that the exact solution is known.

Outputs are views of the library's spinors in device memory.  Their layout: the complex
components colour * 4 + spin in pairs (FP32: float4 [6][V]) or singly (FP64: double2
[12][V]), sites ordered block by block, x fastest inside a block and over the blocks;
even/odd spinors in the same component order over h = x/2 + (Lx/2)(y + Ly (z + Lz t)).
"""
import torch

import qws_amd as Q

PREC = {"f64": Q.F64, "f32": Q.F32}


def _case(op, L, B=(4, 4, 4, 4), **more):
    c = {"op": op, "lx": L[0], "ly": L[1], "lz": L[2], "lt": L[3], "bx": B[0], "by": B[1], "bz": B[2], "bt": B[3],
         "prec": "f32", "links": 12, "kappa": 0.125}
    if op in ("prec_ddd", "solve"):
        c.update(nsap=2, nm=6)
    if op == "solve":
        c.update(nrhs=1, sap="f32", kappa=0.13)
    c.update(more)
    return c


def listed():
    return [
        # the operator on the smallest lattice that is served: a call is one short launch
        _case("dslash", (8, 8, 8, 8), name="dslash_f32_8c8"),
        # the operator on the benchmark lattice, in FP32 (12-real links) ...
        _case("dslash", (32, 32, 32, 64), name="dslash_f32_32c64"),
        # ... and in FP64, the outer solver's operator, on the middle served lattice
        _case("dslash", (24, 24, 24, 48), prec="f64", links=18, name="dslash_f64_24c48"),
        # the inner solver's operator on the benchmark lattice and with its settings: the
        # kernels that most of a solve's time goes to
        _case("prec_ddd", (32, 32, 32, 64), name="sap_f32_32c64"),
        # the same with QWS's default settings on the smallest served lattice
        _case("prec_ddd", (8, 8, 8, 8), nsap=4, nm=2, name="sap_f32_8c8"),
        # 18-real links: what a drop-in caller with links that need not be SU(3) gets
        _case("prec_ddd", (16, 16, 16, 32), nsap=4, nm=2, links=18, name="sap_f32_r18_16c32"),
        # QWS's own domains, the two x halves of one rank's lattice, with extents that
        # are not powers of two: what a drop-in caller gets without choosing blocks
        _case("prec_ddd", (32, 12, 12, 10), (16, 12, 12, 10), nsap=4, nm=2, links=18, name="sap_f32_qws_halves"),
        # the even/odd operator on the benchmark lattice
        _case("mtilde", (32, 32, 32, 64), name="mtilde_f32_32c64"),
        # an even/odd solve on the middle served lattice
        _case("eo_solve", (24, 24, 24, 48), prec="f64", links=18, name="eo_solve_24c48"),
        # a plain solve on the benchmark lattice with its settings
        _case("solve", (32, 32, 32, 64), kappa=0.1365, name="solve_32c64"),
        # twelve right-hand sides (a propagator's spin-colour sources) in one batch
        _case("solve", (16, 16, 16, 32), nrhs=12, name="solve_12rhs_16c32"),
        # the half-precision SAP method (its first sweep is left out: nsap = 3 runs two)
        _case("solve", (24, 24, 24, 48), nsap=3, sap="f16", name="solve_f16sap_24c48"),
    ]


def _extents(rng, step, lo, hi, most):
    """Four multiples of `step`, their volume spread over its logarithm, at most `most`."""
    while True:
        target = (lo ** 4) * (most / lo ** 4) ** rng.random()
        L = [step * max(lo // step, round(target ** 0.25 * 2 ** rng.uniform(-0.7, 0.7) / step)) for _ in range(4)]
        if max(L) <= hi and L[0] * L[1] * L[2] * L[3] <= most:
            return L


def draw(rng):
    c = _draw(rng)
    c["kappa"] = round(rng.uniform(0.12, 0.13), 4)
    return c


def _draw(rng):
    big = 32 ** 3 * 64
    op = rng.choice(["dslash", "dslash", "prec_ddd", "prec_ddd", "prec_ddd", "mtilde", "eo_solve", "solve", "solve"])
    if op == "dslash":
        prec = rng.choice(["f32", "f64"])
        links = 18 if prec == "f64" else rng.choice([12, 18])
        if rng.random() < 0.7:
            return _case(op, _extents(rng, 8, 8, 64, big), prec=prec, links=links)
        L = [2 * rng.randint(4, 20)] + [rng.randint(3, 24) for _ in range(3)]
        return _case(op, L, [L[0] // 2] + L[1:], prec=prec, links=links)
    if op == "prec_ddd":
        nsap, nm = rng.choice([(1, 6), (2, 6), (2, 4), (4, 2), (3, 5)])
        if rng.random() < 0.75:
            return _case(op, _extents(rng, 8, 8, 64, big), nsap=nsap, nm=nm, links=rng.choice([12, 12, 18]))
        L = [2 * rng.randint(4, 20)] + [rng.randint(3, 20) for _ in range(3)]
        return _case(op, L, [L[0] // 2] + L[1:], nsap=nsap, nm=nm, links=18)
    if op == "mtilde":
        prec = rng.choice(["f32", "f64"])
        return _case(op, _extents(rng, 8, 8, 64, big), prec=prec, links=18 if prec == "f64" else rng.choice([12, 18]))
    if op == "eo_solve":
        return _case(op, _extents(rng, 8, 8, 48, 24 ** 3 * 48), prec="f64", links=18)
    sap = rng.choice(["f32", "f32", "f16"])
    nrhs = rng.choice([1, 1, 3, 12])
    return _case(op, _extents(rng, 8, 8, 48, 24 ** 3 * 48 // nrhs), nrhs=nrhs, sap=sap, nsap=3 if sap == "f16" else 2,
                 nm=rng.choice([4, 6]))


# ------------------------------------------------------------------ inputs
def _dims(c):
    L, B = [c["lx"], c["ly"], c["lz"], c["lt"]], [c["bx"], c["by"], c["bz"], c["bt"]]
    return L, B, L[0] * L[1] * L[2] * L[3]


def _cross(a, b):
    return torch.stack([a[:, 1] * b[:, 2] - a[:, 2] * b[:, 1], a[:, 2] * b[:, 0] - a[:, 0] * b[:, 2],
                        a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0]], 1)


def _gauss(gen, *shape):
    return torch.randn(*shape, 2, generator=gen, dtype=torch.float64, device="cuda")


def _fields(c, gen):
    """Links (4, V, 3, 3) complex and packed clover inverse (V, 2, 36), lexicographic sites."""
    V = _dims(c)[2]
    U = torch.empty(4, V, 3, 3, dtype=torch.complex128, device="cuda")
    for mu in range(4):
        h = torch.view_as_complex(_gauss(gen, V, 3, 3))
        m = torch.eye(3, device="cuda") + 0.15j * (h + h.conj().transpose(1, 2))
        r0 = m[:, 0] / torch.linalg.vector_norm(m[:, 0], dim=1, keepdim=True)
        r1 = m[:, 1] - (r0.conj() * m[:, 1]).sum(1, keepdim=True) * r0
        r1 = r1 / torch.linalg.vector_norm(r1, dim=1, keepdim=True)
        U[mu] = torch.stack([r0, r1, _cross(r0, r1).conj()], 1)
    C = 0.02 * torch.randn(V, 2, 36, generator=gen, dtype=torch.float64, device="cuda")
    C[:, :, :6] += 0.5
    return U, C


def _inputs(c, seed):
    """(links, clover, spinors): the spinors are the operand, or the exact solutions of a solve."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    U, C = _fields(c, gen)
    n, V = c.get("nrhs", 1), _dims(c)[2]
    return U, C, [torch.view_as_complex(_gauss(gen, V, 3, 4)) for _ in range(n)]


# ------------------------------------------------------------------ the operators in 64 bits
_g = torch.zeros(4, 4, 4, dtype=torch.complex128)
_g[0, 0, 3], _g[0, 1, 2], _g[0, 2, 1], _g[0, 3, 0] = 1j, 1j, -1j, -1j
_g[1, 0, 3], _g[1, 1, 2], _g[1, 2, 1], _g[1, 3, 0] = 1, -1, -1, 1
_g[2, 0, 2], _g[2, 1, 3], _g[2, 2, 0], _g[2, 3, 1] = 1j, -1j, -1j, 1j
_g[3] = torch.diag(torch.tensor([1, 1, -1, -1], dtype=torch.complex128))


class _Operator:
    """D = 1 - kappa T^-1 H in plain torch, complex128, antiperiodic in t; spinors (V, 3, 4)."""

    def __init__(self, c, U, C):
        self.L, self.B, self.V = _dims(c)
        self.kappa, self.U = c["kappa"], U
        self.A = torch.zeros(self.V, 2, 6, 6, dtype=torch.complex128, device="cuda")
        for r in range(6):
            self.A[:, :, r, r] = C[:, :, r] + 0j
        p = 6
        for r in range(6):
            for k in range(r + 1, 6):
                self.A[:, :, r, k] = torch.complex(C[:, :, p], C[:, :, p + 1])
                self.A[:, :, k, r] = self.A[:, :, r, k].conj()
                p += 2
        i = torch.arange(self.V, device="cuda")
        self.x = []
        for m in range(4):
            self.x.append(i % self.L[m])
            i = i // self.L[m]
        self.colour = sum(self.x[m] // self.B[m] for m in range(4)) % 2
        self.g = _g.cuda()
        self.one = torch.eye(4, dtype=torch.complex128, device="cuda")

    def _shift(self, v, mu, d):
        """v at the site one step along mu in direction d."""
        s = v.reshape(self.L[3], self.L[2], self.L[1], self.L[0], -1)
        return torch.roll(s, -d, 3 - mu).reshape(v.shape)

    def hops(self, v, part="all"):
        """The hops of `part`: all, inside the blocks, across their faces."""
        acc = torch.zeros_like(v)
        for mu in range(4):
            for d in (1, -1):
                w = v @ (self.one - d * self.g[mu]).T
                if d > 0:
                    w = self._shift(w, mu, 1)
                    u = self.U[mu]
                    h = sum(u[:, i, :, None] * w[:, i, None, :] for i in range(3))
                else:
                    u = self.U[mu].conj()
                    h = self._shift(sum(u[:, :, i, None] * w[:, i, None, :] for i in range(3)), mu, -1)
                f = torch.ones(self.V, dtype=torch.float64, device="cuda")
                if mu == 3:
                    f[self.x[3] == (self.L[3] - 1 if d > 0 else 0)] = -1
                if part != "all":
                    l = self.x[mu] % self.B[mu] + d
                    inside = (l >= 0) & (l < self.B[mu])
                    f = f * (inside if part == "inside" else ~inside)
                acc += f[:, None, None] * h
        return acc

    def clover(self, v):
        up, lo = v[:, :, 0:2], v[:, :, 2:4]
        y = []
        for k, x in enumerate((up + lo, up - lo)):
            x = x.transpose(1, 2).reshape(self.V, 6)
            z = sum(self.A[:, k, :, i] * x[:, i, None] for i in range(6))
            y.append(z.reshape(self.V, 2, 3).transpose(1, 2))
        return torch.cat([y[0] + y[1], y[0] - y[1]], 2)

    def D(self, v):
        return v - self.kappa * self.clover(self.hops(v))

    def mtilde(self, v):
        return v - self.kappa ** 2 * self.clover(self.hops(self.clover(self.hops(v))))

    def prec_ddd(self, b, nsap, nm):
        """D M_SAP b in the reference's step order (qws.cc:776-926)."""
        k = self.kappa
        improper = any(self.L[m] == self.B[m] for m in range(1, 4))
        on = [(self.colour == c)[:, None, None] for c in (0, 1)]

        def add(y, c, z):
            return torch.where(on[c], y + z, y)

        def hin(v):
            return k * self.clover(self.hops(v, "inside"))

        def hface(v):
            return k * self.clover(self.hops(v, "face"))

        def block_solve(s, q, c):
            x = s
            for _ in range(max(nm, 1)):
                x = s + hin(x)
            return torch.where(on[c], x, q)

        s, q = b.clone(), torch.zeros_like(b)
        for _ in range(nsap):
            for c in (0, 1):
                q = block_solve(s, q, c)
                s = add(s, c, b - q + hin(q))
                s = add(s, 1 - c, hface(q))
        if improper:
            q = torch.where(on[1], torch.zeros_like(q), q)
        q = block_solve(s, q, 0)
        out = torch.where(on[0], q - hin(q), torch.zeros_like(q))
        if improper:
            s = add(s, 1, hface(q))
            q = block_solve(s, q, 1)
            out = add(out, 1, q - hin(q))
            return out - hface(q)
        f = hface(q)
        out, s = add(out, 1, -f), add(s, 1, f)
        q = block_solve(s, q, 1)
        out = add(out, 1, q - hin(q))
        return add(out, 0, -hface(q))


# ------------------------------------------------------------------ layouts
def _block_order(c):
    """The lexicographic site at each position of the device order."""
    L, B, V = _dims(c)
    i = torch.arange(V, device="cuda").reshape(L[3] // B[3], B[3], L[2] // B[2], B[2], L[1] // B[1], B[1],
                                               L[0] // B[0], B[0])
    return i.permute(0, 2, 4, 6, 1, 3, 5, 7).reshape(-1)


def _even_sites(c):
    L, _, V = _dims(c)
    h = torch.arange(V // 2, device="cuda")
    xh, r = h % (L[0] // 2), h // (L[0] // 2)
    y, z, t = r % L[1], r // L[1] % L[2], r // (L[1] * L[2])
    return 2 * xh + (y + z + t) % 2 + L[0] * r


def _sites(c):
    return _even_sites(c) if c["op"] in ("mtilde", "eo_solve") else _block_order(c)


def _device_layout(c, v, prec):
    w = 4 if prec == "f32" else 2
    return torch.view_as_real(v[_sites(c)]).reshape(-1, 24 // w, w).permute(1, 0, 2).contiguous()


class _DeviceSpinor:
    """A library spinor as an array in device memory; keeps it alive."""

    def __init__(self, spinor, sites, prec):
        w = 4 if prec == "f32" else 2
        self.spinor = spinor
        self.__cuda_array_interface__ = {"shape": (24 // w, sites, w), "typestr": "<f4" if prec == "f32" else "<f8",
                                         "data": (spinor.ptr.value, False), "version": 2}


def _view(spinor, sites, prec):
    return torch.as_tensor(_DeviceSpinor(spinor, sites, prec), device="cuda")


def _host(v):
    return torch.view_as_real(v).cpu().numpy()


# ------------------------------------------------------------------ the cases
def prepare(case, seed):
    c = case
    L, B, V = _dims(c)
    op, prec, eo = c["op"], c["prec"], c["op"] in ("mtilde", "eo_solve")
    U, C, vs = _inputs(c, seed)
    if op in ("solve", "eo_solve"):
        D = _Operator(c, U, C)
        if eo:  # the exact solution and its source live on the even sites
            full = torch.zeros_like(vs[0])
            at = _even_sites(c)
            full[at] = vs[0][at]
            vs = [D.mtilde(full)]
        else:
            vs = [D.D(v) for v in vs]
        del D
    lat = Q.Lattice(L, B, -1, c["links"], kappa=c["kappa"])
    if prec == "f32" and op != "solve":
        lat.load_gauge_f32(torch.view_as_real(U).to(torch.float32).cpu().numpy())
        lat.load_clover_f32(C.to(torch.float32).cpu().numpy())
    else:
        lat.load_gauge(_host(U))
        lat.load_clover(C.cpu().numpy())
    del U, C
    st = {"case": c, "lat": lat}
    if eo:
        lat.eo_from_lattice()
        st["in"] = lat.eo_spinor(PREC[prec], _host(vs[0][_even_sites(c)]))
        st["out"] = lat.eo_spinor(PREC[prec])
        st["views"] = [_view(st["out"], V // 2, prec)]
    elif op == "solve":
        st["in"] = [lat.spinor(Q.F64, _host(v)) for v in vs]
        st["out"] = [lat.spinor(Q.F64) for _ in vs]
        st["views"] = [_view(x, V, "f64") for x in st["out"]]
    else:
        st["in"] = lat.spinor(PREC[prec], _host(vs[0]))
        st["out"] = lat.spinor(PREC[prec])
        st["views"] = [_view(st["out"], V, prec)]
    del vs
    torch.cuda.synchronize()
    torch.cuda.empty_cache()  # the library allocates its device memory itself
    return st


def run(state):
    c, lat, a, o = state["case"], state["lat"], state["in"], state["out"]
    if c["op"] == "dslash":
        lat.dslash(o, a)
    elif c["op"] == "prec_ddd":
        lat.prec_ddd(o, a, c["nsap"], c["nm"])
    elif c["op"] == "mtilde":
        lat.mtilde(o, a)
    elif c["op"] == "eo_solve":
        state["views"][0].zero_()
        lat.eo_bicgstab(o, a, maxiter=2000, tol=1e-12)
    else:
        for x in o:
            x.zero()
        p = dict(nsap=c["nsap"], nm=c["nm"], tol=1e-11, maxiter=40, tol_s=1e-3, maxiter_s=80, true_tol=1e-10,
                 max_restarts=4, sap_precision=Q.F16 if c["sap"] == "f16" else Q.F32)
        if len(o) == 1:
            lat.solve(o[0], a[0], **p)
        else:
            lat.solve_batch(o, a, **p)
    return state["views"]


def exact(case, seed):
    c = case
    U, C, vs = _inputs(c, seed)
    if c["op"] == "solve":
        return [_device_layout(c, v, "f64") for v in vs]
    if c["op"] == "eo_solve":
        return [_device_layout(c, vs[0], "f64")]
    if c["prec"] == "f32":  # the library is given these inputs in 32 bits
        U, C = U.to(torch.complex64).to(torch.complex128), C.float().double()
        vs = [v.to(torch.complex64).to(torch.complex128) for v in vs]
    D = _Operator(c, U, C)
    if c["op"] == "dslash":
        out = D.D(vs[0])
    elif c["op"] == "prec_ddd":
        out = D.prec_ddd(vs[0], c["nsap"], c["nm"])
    else:
        full = torch.zeros_like(vs[0])
        at = _even_sites(c)
        full[at] = vs[0][at]
        out = D.mtilde(full)
    return [_device_layout(c, out, c["prec"])]


# ------------------------------------------------------------------ compulsory work
# flops per site: a hop along x, y, z 168 (projection 12, link times two colour vectors
# 132, sum 24), along t 144; the clover inverse 552; an update with a factor 48
HOPS, CLOVER, UPDATE = 2 * (3 * 168 + 144), 552, 48


def work(case):
    c = case
    _, B, V = _dims(c)
    op, e = c["op"], 8 if c["prec"] == "f64" else 4
    fields = (4 * c["links"] + 72) * e
    d_flops = HOPS + CLOVER + UPDATE
    if op == "dslash":
        return {"bytes": V * (fields + 48 * e), "flops": V * d_flops}
    if op == "mtilde":
        return {"bytes": V * (fields + 24 * e), "flops": V * d_flops}
    if op == "eo_solve":  # about 33 iterations of two operator applications
        return {"bytes": V * (fields + 24 * e), "flops": V * 33 * 2 * d_flops}
    hop = [168, 168, 168, 144]
    face = sum(2 * hop[m] / B[m] for m in range(4))
    inside = HOPS - face + CLOVER + UPDATE
    sap = (c["nsap"] + 1) * ((c["nm"] + 1) * inside + face + CLOVER + UPDATE)
    if op == "prec_ddd":
        return {"bytes": V * (fields + 48 * 4), "flops": V * sap}
    # inner iterations of two preconditioned operators for each source: about 7 at kappa
    # 0.12, 12 at 0.13, 28 at 0.1365
    n = 0.14 / (0.1414 - c["kappa"])
    return {"bytes": V * (72 * 2 * 8 + fields + c["nrhs"] * 48 * 8), "flops": V * c["nrhs"] * n * 2 * sap}
