"""The CG residual step in the epilogue of M^dag's last hop (CLOV_NRR), at the
shapes whose launch rule differs from the other hops'."""
import re

import numpy as np
import pytest

import cps_public_amd as C
from cps_public_amd import fields as F
from tests.helpers import rel, wilson_gauge

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,nrhs", [([4, 4, 4, 4], 3), ([8, 4, 4, 4], 1), ([6, 6, 6, 6], 2)])
def test_two_slice_domain_wall_solve(oracle, L, nrhs):
    """Domain-wall fields of two slices hold one element per site, as the 4-D
    operators do, but their |r|^2 partials are per block (256, 512 and 1296
    elements per rhs: one, two and six blocks, the last of the six a part).
    FP64: the oracle's solution after the same iterations (1e-10, as the
    parity tests).  Mixed: the FP64 stopping rule, and twice its 1e-10 times
    the condition of M^dag M (below 20 on these fields) as the distance."""
    ls, mass = 2, 0.1
    n = int(np.prod(L)) // 2 * ls
    u = wilson_gauge(L, 0.2, 41)
    op = C.make_op(C.OP_DWF, mass=mass, m5=1.8)
    lat = C.Lattice(L, ls, (0, 0, 0, 1))
    lat.import_gauge(u)
    src = np.concatenate([F.gaussian_fermion(n, 42 + k) * (1.0 + 3.0 * k) for k in range(nrhs)])
    sol, res = lat.invcg(op, src, C.make_cg_arg(1e-10, 2000), nrhs=nrhs)
    half, hres = lat.invcg(op, src, C.make_cg_arg(1e-10, 2000, precision=C.PREC_MIXED_HALF), nrhs=nrhs)
    lat.close()
    d = oracle.dwf_struct(L, ls, 1.8)
    for k in range(nrhs):
        part = slice(24 * n * k, 24 * n * (k + 1))
        x, it, _ = oracle.dwf_invcg(u, src[part], mass, 1e-10, 2000, d)
        assert abs(res[k].iterations - it) <= 1
        assert res[k].true_res <= 1.1e-10 and rel(sol[part], x) < 1e-10
        assert hres[k].true_res <= 1e-10 and rel(half[part], x) < 4e-9


def _flags(err):
    """Launch flags of the residual steps reported on stderr."""
    return [int(m) for m in re.findall(r"residual step -> block \d+ flags (\d+)", err)]


RHSGROUP = 32   # HOP_RHSGROUP


@pytest.mark.parametrize("L,nrhs", [([4, 4, 8, 4], 4), ([8, 8, 4, 4], 4), ([6, 6, 4, 6], 2), ([10, 4, 6, 6], 4),
                                    ([6, 6, 6, 6], 4), ([6, 10, 6, 6], 6), ([14, 14, 10, 14], 14)])
def test_residual_step_mappings(monkeypatch, capfd, L, nrhs):
    """Wilson solves with the hops, the residual step among them, in element
    order and with 4 or 2 rhs of a site in a wavefront (CPS_HIP_HOP_MODE):
    whole and part chunks of 64 sites (256, 512, 432, 720, 648, 1080 and 13720
    sites a parity), groups in blocks of 256 (4 and 2 rhs) and of 128 (the first
    and the fourth case), the last one large enough for streaming stores.  FP64: an element's arithmetic and the tree
    of the partial sums are the same, so are all bits.  Half precision: the
    two mappings are separate compilations (a few FP32 results round
    differently), so twice the stopping rule's 1e-10 times the condition of
    M^dag M, which is 20 for 6^4 and below 100 at this mass."""
    u = wilson_gauge(L, 0.2, 71)
    n = int(np.prod(L)) // 2
    op = C.make_op(C.OP_WILSON, mass=0.1)
    src = np.concatenate([F.gaussian_fermion(n, 72 + k) * (1.0 + k) for k in range(nrhs)])
    monkeypatch.setenv("CPS_HIP_TUNE_REPORT", "1")
    monkeypatch.setenv("CPS_HIP_RHS_WINDOW", "0")   # (a shrunk window may hold an odd count, which no group divides)
    out = {}
    for mode in ("element", "rhsgroup"):
        monkeypatch.setenv("CPS_HIP_HOP_MODE", mode)
        lat = C.Lattice(L, 1, (0, 0, 0, 1))
        lat.import_gauge(u)
        capfd.readouterr()
        out[mode] = [lat.invcg(op, src, C.make_cg_arg(1e-10, 1000, precision=p), nrhs=nrhs)
                     for p in (C.PREC_DOUBLE, C.PREC_MIXED_HALF)]
        flags = _flags(capfd.readouterr().err)
        assert flags and all(((f & RHSGROUP) != 0) == (mode == "rhsgroup") for f in flags), flags
        lat.close()
    (xe, re_), (xg, rg) = out["element"][0], out["rhsgroup"][0]
    assert [r.iterations for r in re_] == [r.iterations for r in rg]
    assert np.array_equal(xe, xg)
    (xe, re_), (xg, rg) = out["element"][1], out["rhsgroup"][1]
    assert max(r.true_res for r in re_ + rg) <= 1e-10
    for k in range(nrhs):
        part = slice(24 * n * k, 24 * n * (k + 1))
        assert rel(xg[part], xe[part]) < 2e-8


@pytest.mark.parametrize("kind", ["wilson", "dwf", "mobius", "clover"])
@pytest.mark.parametrize("graph", [1, 0])
def test_fp64_lagged_steps(monkeypatch, kind, graph):
    """FP64 solves whose rhs converge at different iterations (the first and
    the last start close to their solutions, so the window of active rhs
    shrinks at both ends, where pending solution steps are applied).
    CPS_HIP_LAGGED_X=0 with the residual step a pass of its own: the same
    arithmetic, so the same bits.  CPS_HIP_R_IN_HOP=0: the same for the
    operators without that step; for Wilson and domain wall |r|^2 is the sum
    of other partials, so twice the stopping rule's 1e-10 times the condition
    of M^dag M (21 and 60 on these fields), and the iterations to one."""
    L, nrhs, kappas = [4, 4, 4, 8], 4, [0.130, 0.1325]
    ls = 8 if kind in ("dwf", "mobius") else 1
    op = {"wilson": C.make_op(C.OP_WILSON, mass=0.1), "dwf": C.make_op(C.OP_DWF, mass=0.1, m5=1.8),
          "mobius": C.make_op(C.OP_MOBIUS, mass=0.1, m5=1.8, b=1.5, c=0.5),
          "clover": C.make_op(C.OP_CLOVER, mass=1.0 / (2 * kappas[0]) - 4.0, csw=1.0)}[kind]
    n = int(np.prod(L)) // 2 * ls
    src = np.concatenate([F.gaussian_fermion(n, 91 + k) for k in range(nrhs)])
    lat = C.Lattice(L, ls, (0, 0, 0, 1))
    lat.import_gauge(wilson_gauge(L, 0.2, 90))
    if kind == "clover":
        lat.clover_build(kappas, 1.0)
    guess = np.zeros_like(src)
    near, _ = lat.invcg(op, src, C.make_cg_arg(1e-5, 1000), nrhs=nrhs)
    for k in (0, nrhs - 1):
        guess[24 * n * k:24 * n * (k + 1)] = near[24 * n * k:24 * n * (k + 1)]
    arg = C.make_cg_arg(1e-10, 1000)
    arg.check_every, arg.use_graph = 3, graph
    out = {}
    for lagged, in_hop in (("1", "1"), ("1", "0"), ("0", "0"), ("0", "1")):
        monkeypatch.setenv("CPS_HIP_LAGGED_X", lagged)
        monkeypatch.setenv("CPS_HIP_R_IN_HOP", in_hop)
        x, res = lat.invcg(op, src, arg, guess=guess, nrhs=nrhs)
        out[lagged + in_hop] = (x, [r.iterations for r in res], max(r.true_res for r in res))
    lat.close()
    x, its, _ = out["00"]
    assert max(its[0], its[-1]) + 3 < min(its[1:-1])
    assert max(o[2] for o in out.values()) <= 1.1e-10
    for same in ("10", "01") + (("11",) if kind in ("mobius", "clover") else ()):
        assert np.array_equal(out[same][0], x) and out[same][1] == its
    assert all(abs(a - b) <= 1 for a, b in zip(out["11"][1], its))
    assert all(rel(out["11"][0][p], x[p]) < 1.2e-8 for p in (slice(24 * n * k, 24 * n * (k + 1)) for k in range(nrhs)))
