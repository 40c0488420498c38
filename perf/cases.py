"""Performance cases: the work that a user of this library has it do.

The library inverts even-odd preconditioned Wilson, domain-wall, Moebius and
clover operators.  Most of its time goes into batched conjugate-gradient
solves of M^dag M x = b on vectors that stay in device memory
(cps_hip_invcg_device): in FP64, or in a mixed mode (FP16, BF16-link or FP32
iterations with FP64 reliable updates).  Beside them stand the calls that take
host vectors as CPS's own fermion library does: a hop, an operator
application, a solve and a 12-source point propagator.

Gauge links are exp(i eps H) with H traceless Hermitian Gaussian, re-unitarised,
antiperiodic in t, as the benchmark and the tests use them; sources are
Gaussian or spin-colour points.  Solves stop at 1e-12, the tolerance of the
solver tests.
"""
import ctypes

import numpy as np
import torch

import cps_public_amd as C

KIND = {"wilson": C.OP_WILSON, "dwf": C.OP_DWF, "mobius": C.OP_MOBIUS, "clover": C.OP_CLOVER}
PREC = {"double": C.PREC_DOUBLE, "half": C.PREC_MIXED_HALF, "bf16": C.PREC_MIXED_BF16, "single": C.PREC_MIXED_SINGLE}
M5, MOBIUS_B, MOBIUS_C, CSW = 1.8, 1.5, 0.5, 1.0
STOP = 1e-12
TEMPORAL_BC = (0, 0, 0, 1)


def _case(name, call, op, prec, L, ls=1, nrhs=1, mass=0.02, eps=0.2, kappas=1, source="gauss"):
    return {"name": name, "call": call, "op": op, "prec": prec, "x": L[0], "y": L[1], "z": L[2], "t": L[3],
            "ls": ls, "nrhs": nrhs, "mass": mass, "eps": eps, "kappas": kappas, "source": source}


def listed():
    return [
        # one library call on a parity-test lattice: what a CPS run on a small
        # lattice issues one by one (wilson_dslash on host vectors)
        _case("dslash_wilson_8x8x8x8", "dslash", "wilson", "double", (8, 8, 8, 8), eps=0.3),
        # one domain-wall M^dag M on host vectors (dwf_mdagm), the library call
        # of an unmodified CPS solver or eigensolver
        _case("mdagm_dwf_16x16x16x32_ls16", "mdagm", "dwf", "double", (16, 16, 16, 32), ls=16, mass=0.01),
        # the smallest solve in use: InvCg on host vectors, a few dozen short
        # iterations of a lattice that fits any cache
        _case("cg_wilson_8x8x8x8_double", "invcg", "wilson", "double", (8, 8, 8, 8), mass=0.16666, eps=0.3),
        # the small lattice of the solve-serving stream: all 12 point sources
        # of one domain-wall propagator
        _case("cg_dwf_8x8x8x8_ls8_half_x12", "solve", "dwf", "half", (8, 8, 8, 8), ls=8, nrhs=12, mass=0.02,
              source="point"),
        # a Wilson propagator on the middle lattice of that stream
        _case("cg_wilson_16x16x16x32_half_x12", "solve", "wilson", "half", (16, 16, 16, 32), nrhs=12, mass=0.05,
              source="point"),
        # one domain-wall source at a time, mixed and in FP64 (force and
        # measurement solves; the bench's Shamir workload)
        _case("cg_dwf_16x16x16x32_ls16_half", "solve", "dwf", "half", (16, 16, 16, 32), ls=16, mass=0.01),
        _case("cg_dwf_16x16x16x32_ls16_double", "solve", "dwf", "double", (16, 16, 16, 32), ls=16, mass=0.01),
        # the largest: a Moebius propagator, 12 point sources in one solve
        _case("cg_mobius_16x16x16x32_ls16_half_x12", "solve", "mobius", "half", (16, 16, 16, 32), ls=16, nrhs=12,
              mass=0.02, source="point"),
        # uneven extents, an Ls that is no power of two, an odd batch, BF16 links
        _case("cg_mobius_10x12x14x18_ls12_bf16_x5", "solve", "mobius", "bf16", (10, 12, 14, 18), ls=12, nrhs=5,
              mass=0.05),
        # clover propagators at two kappas, solved together
        _case("cg_clover_24x24x24x48_half_x24", "solve", "clover", "half", (24, 24, 24, 48), nrhs=24, mass=-0.3182,
              eps=0.15, kappas=2, source="point"),
        # Moebius on a large spatial volume with few sources
        _case("cg_mobius_24x24x24x32_ls16_half_x2", "solve", "mobius", "half", (24, 24, 24, 32), ls=16, nrhs=2,
              mass=0.05),
        # a whole measurement call: point propagator of 12 sources, host output
        _case("propagator_wilson_16x16x16x32_double", "propagator", "wilson", "double", (16, 16, 16, 32), nrhs=12,
              mass=0.05, source="point"),
    ]


def draw(rng):
    """Another case of the listed ranges: operators, precisions, uneven even
    extents, any even Ls from 4 to 24, 1 to 16 right-hand sides."""
    while True:
        op = rng.choice(("wilson", "dwf", "mobius", "clover"))
        call = rng.choice(("solve", "solve", "solve", "solve", "solve", "invcg", "mdagm", "dslash", "propagator"))
        prec = rng.choice(("half", "half", "bf16", "single", "double"))
        L = tuple(2 * rng.randint(3, 9) for _ in range(3)) + (2 * int(round(2 ** rng.uniform(2, 4))),)
        ls = rng.choice((4, 6, 8, 10, 12, 16, 16, 20, 24)) if op in ("dwf", "mobius") else 1
        nrhs, kappas = int(round(2 ** rng.uniform(0, 4))), 1
        mass, eps = round(10 ** rng.uniform(-2, -1), 4), rng.choice((0.15, 0.2, 0.25))
        if call == "dslash":
            op, prec, nrhs, ls = "wilson", "double", 1, 1
        if call == "mdagm":
            prec, nrhs = "double", min(nrhs, 2)
        if call == "propagator":
            op, nrhs, ls = "wilson", 12, 1
        if op == "wilson":
            mass = round(mass + 0.05, 4)
        if op == "clover":
            mass, eps, kappas = round(-0.3 + mass, 4), 0.15, rng.choice((1, 2))
            nrhs += nrhs % kappas
        c = _case("", call, op, prec, L, ls, nrhs, mass, eps, kappas, rng.choice(("gauss", "point")))
        del c["name"]
        w = work(c)
        if w["bytes"] < 0.4 * work(listed()[7])["bytes"] * (1.0 if prec != "double" else 0.7):
            return c


# ---- sizes -------------------------------------------------------------------

def _extents(c):
    return [c["x"], c["y"], c["z"], c["t"]]


def _vcb(c):
    return c["x"] * c["y"] * c["z"] * c["t"] // 2


def _slices(c):
    return c["ls"] if c["op"] in ("dwf", "mobius") else 1


def _kappas(c):
    """The kappa list of a clover case: the mass's own, then heavier ones."""
    k0 = 1.0 / (2 * (c["mass"] + 4.0))
    return [k0 * (1.0 - 0.004 * i) for i in range(c["kappas"])]


def _iterations(c):
    """CG iterations to the tolerance, estimated from counts seen on such
    fields: at these masses they grow with the lattice's linear extent."""
    per = {"wilson": 6.5, "clover": 5.0, "dwf": 11.0, "mobius": 15.5}[c["op"]]
    return per * (2.0 * _vcb(c)) ** 0.25


def work(c):
    """Compulsory traffic: every link once and every spinor once in and once
    out for each hop, in the format that the hop computes on; per iteration of
    a solve four hops and one pass in and out over x, r and p; FP64 vectors of
    the caller once.  1320 flops a hop and spinor, 48 a fifth-dimension term."""
    spin = {"double": 192.0, "single": 96.0}.get(c["prec"], 52.0)
    link = {"double": 144.0, "single": 48.0}.get(c["prec"], 36.0)
    v, n = 2.0 * _vcb(c), float(_vcb(c) * _slices(c) * c["nrhs"])
    hop = 4 * v * link + 2 * n * spin
    clover = 2 * 2 * _vcb(c) * c["kappas"] * 72 * spin / 24 if c["op"] == "clover" else 0.0
    flops = n * (1320 + (48 if _slices(c) > 1 else 0) + (504 if c["op"] == "clover" else 0))
    ends = 2 * n * 192.0
    if c["call"] == "dslash":
        return {"bytes": hop, "flops": flops}
    if c["call"] == "mdagm":
        return {"bytes": 2 * n * spin + 4 * v * link, "flops": 4 * flops}
    it = _iterations(c)
    if c["call"] == "propagator":
        ends = v * 288 * 8
    return {"bytes": it * (4 * hop + clover + 6 * n * spin) + ends, "flops": it * (4 * flops + n * 144)}


# ---- inputs ------------------------------------------------------------------

def _generator(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 16 + stream)
    return g


def _mul3(a, b):
    return sum(a[..., :, k, None] * b[..., None, k, :] for k in range(3))


def _links(c, seed):
    """[t][z][y][x][mu][3][3] SU(3) links exp(i eps H), without boundary signs."""
    n = 8 * _vcb(c)
    h = torch.view_as_complex(torch.randn(n, 3, 3, 2, dtype=torch.float64, device="cuda", generator=_generator(seed, 1)))
    h = 0.5 * (h + h.conj().transpose(1, 2))
    h -= (h.diagonal(dim1=1, dim2=2).sum(1) / 3)[:, None, None] * torch.eye(3, dtype=h.dtype, device=h.device)
    h *= 1j * c["eps"]
    u = torch.eye(3, dtype=h.dtype, device=h.device).expand(n, 3, 3).clone()
    for k in range(8, 0, -1):   # Horner form of the exponential's series
        u = torch.eye(3, dtype=h.dtype, device=h.device) + _mul3(h, u) / k
    r0 = u[:, 0] / u[:, 0].norm(dim=1, keepdim=True)
    r1 = u[:, 1] - (r0.conj() * u[:, 1]).sum(1, keepdim=True) * r0
    r1 = r1 / r1.norm(dim=1, keepdim=True)
    r2 = torch.linalg.cross(r0, r1).conj()
    return torch.stack([r0, r1, r2], 1).reshape(c["t"], c["z"], c["y"], c["x"], 4, 3, 3)


def _sources(c, seed):
    """nrhs checkerboard vectors in the order the library takes, on the GPU."""
    per = 24 * _vcb(c) * _slices(c)
    g = _generator(seed, 2)
    if c["source"] == "gauss":
        return torch.randn(c["nrhs"], per, dtype=torch.float64, device="cuda", generator=g)
    b = torch.zeros(c["nrhs"], per, dtype=torch.float64, device="cuda")
    site = int(torch.randint(_vcb(c), (1,), device="cuda", generator=g))
    k = torch.arange(c["nrhs"], device="cuda")
    b[k, 24 * site + 2 * (k % 12)] = 1.0
    return b


def _point(c, seed):
    g = torch.Generator()
    g.manual_seed(int(seed))
    return [int(torch.randint(n, (1,), generator=g)) for n in _extents(c)]


def _op(c):
    mobius = c["op"] == "mobius"
    return C.make_op(KIND[c["op"]], mass=c["mass"], m5=M5, b=MOBIUS_B if mobius else 1.0,
                     c=MOBIUS_C if mobius else 0.0, csw=CSW)


def prepare(c, seed):
    """A lattice handle with the gauge field (and clover fields) resident, the
    operator and solver arguments, and the sources: on the host for the calls
    that take host vectors, in device memory for the device-resident solve."""
    lat = C.Lattice(_extents(c), _slices(c), TEMPORAL_BC)
    lat.import_gauge_canonical(torch.view_as_real(_links(c, seed)).cpu().numpy().reshape(-1))
    if c["op"] == "clover":
        lat.clover_build(_kappas(c), CSW)
    s = {"case": c, "lat": lat, "op": _op(c),
         "arg": C.make_cg_arg(STOP, 5000, PREC[c["prec"]], reliable_every=100,
                              reliable_delta=0.1 if c["prec"] == "bf16" else 0.03)}
    if c["call"] == "propagator":
        s["point"] = _point(c, seed)
        return s
    b = _sources(c, seed)
    if c["call"] == "solve":
        s["src"], s["sol"] = b, torch.zeros_like(b)
        s["res"] = (C.CgResult * c["nrhs"])()
        torch.cuda.synchronize()
    else:
        s["src"] = b.reshape(-1).cpu().numpy()
    return s


def run(s):
    c, lat = s["case"], s["lat"]
    if c["call"] == "solve":
        # initial guess 0; the library works on a stream of its own
        s["sol"].zero_()
        torch.cuda.current_stream().synchronize()
        rc = C.lib().cps_hip_invcg_device(lat.h, ctypes.byref(s["op"]), ctypes.c_void_p(s["sol"].data_ptr()),
                                          ctypes.c_void_p(s["src"].data_ptr()), c["nrhs"], ctypes.byref(s["arg"]),
                                          s["res"])
        if rc:
            raise C.CpsHipError(rc, "cps_hip_invcg_device")
        return list(s["sol"].unbind(0))
    if c["call"] == "invcg":
        return list(lat.invcg(s["op"], s["src"], s["arg"], nrhs=c["nrhs"])[0].reshape(c["nrhs"], -1))
    if c["call"] == "propagator":
        return lat.qpropw_point(s["op"], s["point"], s["arg"])[0]
    if c["call"] == "mdagm":
        out, norms = lat.mdagm(s["op"], s["src"], nrhs=c["nrhs"])
        return [out, norms]
    return lat.wilson_dslash(s["src"], 1, 0)


# ---- exact values: the operators and CG in plain torch, 64 bits ----------------

# gamma_mu couples the upper spins to the lower: (1 + A gamma_mu) psi has
# h_0 = psi_0 + A c_0 psi_i0 and h_1 = psi_1 + A c_1 psi_i1
_GAMMA = (((3, 1j), (2, 1j)), ((3, -1.0), (2, 1.0)), ((2, 1j), (3, -1j)), ((2, 1.0), (3, 1.0)))


class _Exact:
    """The operators on checkerboard fields [spin 4][colour 3][site][column],
    columns = rhs x slices (slices fastest)."""

    def __init__(self, c, seed, nrhs):
        self.c, self.nrhs, self.ls = c, nrhs, _slices(c)
        Lx, Ly, Lz, Lt = _extents(c)
        u = _links(c, seed)
        u[Lt - 1, :, :, :, 3] *= -1
        t, z, y, x = torch.meshgrid(*(torch.arange(n, device="cuda") for n in (Lt, Lz, Ly, Lx)), indexing="ij")
        par = (x + y + z + t) % 2
        site = x // 2 + (Lx // 2) * (y + Ly * (z + Lz * t))
        v = _vcb(c)
        flat = lambda a: a.reshape(-1)   # noqa: E731
        where = torch.empty(2, v, dtype=torch.long, device="cuda")   # full-lattice position of a checkerboard site
        full = torch.arange(2 * v, device="cuda")
        where[flat(par), flat(site)] = full
        u = u.reshape(2 * v, 4, 3, 3)
        self.u, self.where, self.extents = u, where, (Lt, Lz, Ly, Lx)
        self.nbr, self.mat = {}, {}
        for mu, axis in enumerate((3, 2, 1, 0)):
            for d in (0, 1):
                n = torch.roll(full.reshape(Lt, Lz, Ly, Lx), 1 if d else -1, axis).reshape(-1)
                for p in (0, 1):
                    there = n[where[p]]
                    self.nbr[p, mu, d] = flat(site)[there]
                    m = u[there, mu].conj().transpose(1, 2) if d else u[where[p], mu]
                    self.mat[p, mu, d] = m.permute(1, 2, 0).contiguous()[..., None]
        self.kappas = torch.tensor(_kappas(c) if c["op"] == "clover" else [1.0 / (2 * (c["mass"] + 4.0))],
                                   dtype=torch.float64, device="cuda")
        if self.ls > 1:
            one, m = torch.eye(self.ls, dtype=torch.float64, device="cuda"), c["mass"]
            down = torch.roll(one, 1, 0)   # row s takes slot s-1
            down[0, -1] = -m
            up = torch.roll(one, -1, 0)
            up[-1, 0] = -m
            self.shift = {0: (down, up), 1: (up, down)}
        if c["op"] == "clover":
            self._clover()

    def hop(self, psi, p, dag):
        """The 4-D hop from parity 1-p onto parity p."""
        out = torch.zeros(psi.shape[:2] + (_vcb(self.c),) + psi.shape[3:], dtype=psi.dtype, device=psi.device)
        for mu in range(4):
            (i0, c0), (i1, c1) = _GAMMA[mu]
            for d in (0, 1):
                a = (1 if d else -1) * (-1 if dag else 1)
                for s, i, k in ((0, i0, c0), (1, i1, c1)):
                    h = (psi[s] + (a * k) * psi[i])[:, self.nbr[p, mu, d]]
                    m = self.mat[p, mu, d]
                    for r in range(3):
                        w = m[r, 0] * h[0]
                        w.addcmul_(m[r, 1].expand_as(w), h[1]).addcmul_(m[r, 2].expand_as(w), h[2])
                        out[s, r] += w
                        out[i, r] += (a * np.conj(k)) * w
        return out

    def fifth(self, psi, upper, lower):
        """ls x ls matrices on the slices of the upper and lower spins."""
        n = psi.shape
        f = lambda v, m: (v.reshape(-1, self.ls) @ m.to(v.dtype).T).reshape(v.shape)   # noqa: E731
        return torch.cat([f(psi[:2], upper), f(psi[2:], lower)]).reshape(n)

    def _clover(self):
        Lt, Lz, Ly, Lx = self.extents
        u = self.u.reshape(Lt, Lz, Ly, Lx, 4, 3, 3)
        axis = (3, 2, 1, 0)
        at = lambda mu, *steps: self._rolled(u[..., mu, :, :], axis, steps)   # noqa: E731
        dag = lambda m: m.conj().transpose(-1, -2)   # noqa: E731
        g = torch.zeros(4, 4, 4, dtype=u.dtype, device=u.device)
        for mu, ((i0, c0), (i1, c1)) in enumerate(_GAMMA):
            g[mu, 0, i0], g[mu, 1, i1], g[mu, i0, 0], g[mu, i1, 1] = c0, c1, np.conj(c0), np.conj(c1)
        total = 0
        for m in range(4):
            for n in range(m + 1, 4):
                f = _mul3(_mul3(at(m), at(n, (m, 1))), _mul3(dag(at(m, (n, 1))), dag(at(n))))
                f = f + _mul3(_mul3(at(n), dag(at(m, (m, -1), (n, 1)))), _mul3(dag(at(n, (m, -1))), at(m, (m, -1))))
                f = f + _mul3(_mul3(dag(at(m, (m, -1))), dag(at(n, (m, -1), (n, -1)))),
                              _mul3(at(m, (m, -1), (n, -1)), at(n, (n, -1))))
                f = f + _mul3(_mul3(dag(at(n, (n, -1))), at(m, (n, -1))), _mul3(at(n, (m, 1), (n, -1)), dag(at(m))))
                f = ((f - dag(f)) / 8).reshape(-1, 3, 3)
                comm = g[m] @ g[n] - g[n] @ g[m]
                total = total + (comm[None, :, None, :, None] * f[:, None, :, None, :]).reshape(-1, 12, 12)
        one = torch.eye(12, dtype=u.dtype, device=u.device)
        self.a_oo = [one - 0.5 * float(k) * CSW * total[self.where[1]] for k in self.kappas]
        self.a_ee_inv = [torch.linalg.inv(one - 0.5 * float(k) * CSW * total[self.where[0]]) for k in self.kappas]

    @staticmethod
    def _rolled(f, axis, steps):
        for mu, by in steps:
            f = torch.roll(f, -by, axis[mu])
        return f

    def _block(self, mats, psi):
        per = psi.shape[3] // len(mats)
        v = psi.reshape(12, psi.shape[2], -1).permute(1, 0, 2)
        out = [m @ v[:, :, k * per:(k + 1) * per].contiguous() for k, m in enumerate(mats)]
        return torch.cat(out, 2).permute(1, 0, 2).reshape(psi.shape).contiguous()

    def m(self, psi, dag):
        """The preconditioned operator; a domain-wall field is a pair of
        4-D parities whose other slices are zero."""
        c, op = self.c, self.c["op"]
        if op == "wilson":
            k = float(self.kappas[0])
            return psi - k * k * self.hop(self.hop(psi, 0, dag), 1, dag)
        if op == "clover":
            k2 = (self.kappas ** 2).repeat_interleave(psi.shape[3] // len(self.kappas))
            t = self._block(self.a_ee_inv, self.hop(psi, 0, dag))
            return self._block(self.a_oo, psi) - k2 * self.hop(t, 1, dag)
        up, lo = self.shift[dag]
        if op == "dwf":
            k = 1.0 / (2 * (4 + 1.0 - M5))
            d = lambda f: tuple(self.hop(f[1 - p], p, dag) + 2 * self.fifth(f[p], up, lo) for p in (0, 1))   # noqa: E731
            t = d(d((psi[0], psi[1])))
            return torch.stack([psi[p] - k * k * t[p] for p in (0, 1)])
        kb = 1.0 / (2 * (MOBIUS_B * (4 - M5) + 1.0))
        ratio = kb * 2 * (MOBIUS_C * (4 - M5) - 1.0)
        one = torch.eye(self.ls, dtype=torch.float64, device="cuda")
        m5, bc = [one + ratio * s for s in (up, lo)], [MOBIUS_B * one + MOBIUS_C * s for s in (up, lo)]
        inv = [torch.linalg.inv(a) for a in m5]
        if not dag:
            t = self.fifth(kb * self.hop(self.fifth(psi, *bc), 0, 0), *(b @ a for a, b in zip(inv, bc)))
            return self.fifth(psi, *m5) - kb * self.hop(t, 1, 0)
        t = self.fifth(kb * self.hop(psi, 0, 1), *(a @ b for a, b in zip(inv, bc)))
        return self.fifth(psi, *m5) - kb * self.fifth(self.hop(t, 1, 1), *bc)

    def _dot(self, a, b):
        v = (torch.view_as_real(a) * torch.view_as_real(b)).sum(-1)
        return v.flatten(0, -2).sum(0).reshape(self.nrhs, self.ls).sum(1)

    def _wide(self, a):
        return a.repeat_interleave(self.ls)

    def solve(self, b, stop=2e-14):
        """CG on M^dag M, every rhs with its own scalars, restarted from the
        true residual."""
        x = torch.zeros_like(b)
        goal = stop ** 2 * self._dot(b, b)
        for _ in range(3):
            r = b - self.m(self.m(x, 0), 1)
            p, rr = r.clone(), self._dot(r, r)
            for i in range(4000):
                live = rr > goal
                if i % 10 == 0 and not bool(live.any()):
                    break
                q = self.m(self.m(p, 0), 1)
                alpha = torch.where(live, rr / self._dot(p, q), 0.0)
                x += self._wide(alpha) * p
                r -= self._wide(alpha) * q
                new = self._dot(r, r)
                p = r + self._wide(torch.where(live, new / rr, 0.0)) * p
                rr = torch.where(live, new, rr)
        return x

    # the library's vectors: [rhs][slice][site][spin][colour], odd checkerboard
    def load(self, b):
        f = torch.view_as_complex(b.reshape(self.nrhs, self.ls, -1, 4, 3, 2).contiguous())
        f = f.permute(3, 4, 2, 0, 1).reshape(4, 3, -1, self.nrhs * self.ls).contiguous()
        if self.c["op"] != "dwf":
            return f
        s = torch.arange(self.ls, device="cuda").repeat(self.nrhs)
        return torch.stack([torch.where((s + 1) % 2 == p, f, 0.0) for p in (0, 1)])

    def store(self, f):
        f = f.sum(0) if self.c["op"] == "dwf" else f
        f = f.reshape(4, 3, -1, self.nrhs, self.ls).permute(3, 4, 2, 0, 1).contiguous()
        return torch.view_as_real(f).reshape(self.nrhs, -1)


def _affordable(c):
    """How many right-hand sides the exact solution is worked out for: a few
    seconds of plain torch."""
    each = _vcb(c) * _slices(c) * (2 if c["op"] == "dwf" else 1) * _iterations(c)
    return int(min(c["nrhs"], 4.5e8 // each)) // c["kappas"] * c["kappas"]


def exact(c, seed):
    if c["call"] == "dslash":
        e = _Exact(c, seed, 1)
        return e.store(e.hop(e.load(_sources(c, seed)), 0, 0)).reshape(-1).cpu().numpy()
    if c["call"] == "mdagm":
        e = _Exact(c, seed, c["nrhs"])
        t = e.m(e.load(_sources(c, seed)), 0)
        return [e.store(e.m(t, 1)).reshape(-1).cpu().numpy(), e._dot(t, t).cpu().numpy()]
    if c["call"] == "propagator":
        return _exact_propagator(c, seed)
    n = _affordable(c)
    if c["op"] == "clover" and n < c["nrhs"]:
        n = 0 if n < c["kappas"] else min(n // c["kappas"], c["nrhs"] // c["kappas"])
        one = dict(c, kappas=1)   # the first kappa's rhs
    else:
        one = c
    if n < 1:
        return None
    e = _Exact(one, seed, n)
    x = e.store(e.solve(e.load(_sources(c, seed)[:n])))
    return [x[k] if k < n else None for k in range(c["nrhs"])]


def _exact_propagator(c, seed):
    """Columns of (1 - kappa H)^-1 for the 12 unit sources at the case's point."""
    e = _Exact(c, seed, 12)
    x, y, z, t = _point(c, seed)
    k = float(e.kappas[0])
    v = _vcb(c)
    b = [torch.zeros(4, 3, v, 12, dtype=torch.complex128, device="cuda") for _ in (0, 1)]
    site = x // 2 + (c["x"] // 2) * (y + c["y"] * (z + c["z"] * t))
    for n in range(12):
        b[(x + y + z + t) % 2][n // 3, n % 3, site, n] = 1.0
    odd = e.solve(e.m(b[1] + k * e.hop(b[0], 1, 0), 1))
    even = b[0] + k * e.hop(odd, 0, 0)
    out = torch.empty(2 * v, 4, 3, 12, dtype=torch.complex128, device="cuda")
    out[e.where[0]] = even.permute(2, 0, 1, 3)
    out[e.where[1]] = odd.permute(2, 0, 1, 3)
    return out.reshape(c["t"], c["z"], c["y"], c["x"], 4, 3, 4, 3).cpu().numpy()
