"""The half-precision hop kernels that the launcher picks by itself (SU(3)
products on the matrix cores where a site holds a multiple of 4 slots)
against the general element kernel, over the layouts and epilogues they
accept."""
import numpy as np
import pytest

import cps_public_amd as C
from cps_public_amd import fields as F
from tests.helpers import rel, wilson_gauge

pytestmark = pytest.mark.gpu

# (kind, Ls, lattice, rhs): 4 to 16 slots per site, powers of two and not,
# lattices with and without an 8-way (y, z) split, one and several rhs
CASES = [("dwf", 8, [4, 4, 4, 8], 1), ("dwf", 16, [8, 8, 8, 4], 2), ("dwf", 24, [6, 4, 10, 4], 3),
         ("dwf", 32, [4, 8, 4, 6], 1), ("mobius", 4, [4, 4, 4, 8], 3), ("mobius", 8, [8, 4, 8, 6], 2),
         ("mobius", 12, [10, 4, 6, 4], 1), ("mobius", 16, [4, 4, 4, 4], 2), ("mobius", 16, [8, 8, 4, 6], 1),
         ("mobius", 20, [4, 8, 8, 4], 2)]


@pytest.mark.parametrize("prec", [C.PREC_MIXED_HALF, C.PREC_MIXED_BF16])
@pytest.mark.parametrize("kind,ls,L,nrhs", CASES)
def test_default_half_hop_matches_element_mapping(monkeypatch, kind, ls, L, nrhs, prec):
    """M^dag M and |M x|^2.  Both kernels add the same FP16 products in FP32
    and store every intermediate field in FP16 (four hops, each rounded to
    2^-11 of a site's largest real), so the two results differ by at most one
    rounding step per stored field, and neither is further from the FP64
    operator than the other by more than a fraction of its own error."""
    u = wilson_gauge(L, 0.2, 310)
    op = C.make_op(C.OP_MOBIUS, mass=0.05, m5=1.8, b=1.5, c=0.5) if kind == "mobius" else \
        C.make_op(C.OP_DWF, mass=0.05, m5=1.8)
    n = int(np.prod(L)) // 2 * ls
    src = np.concatenate([F.gaussian_fermion(n, 311 + k) for k in range(nrhs)])
    res = {}
    for mode in ("element", ""):
        monkeypatch.setenv("CPS_HIP_HOP_MODE", mode)
        lat = C.Lattice(L, ls, (0, 0, 0, 1))
        lat.import_gauge(u)
        res[mode] = lat.mdagm_prec(op, src, prec, nrhs=nrhs)
        if not mode:
            exact, norms = lat.mdagm(op, src, nrhs=nrhs)
        lat.close()
    assert rel(res[""][0], res["element"][0]) < 4 * 2.0 ** -11
    assert np.allclose(res[""][1], res["element"][1], rtol=2.0 ** -11, atol=0)
    err = {m: rel(res[m][0], exact) for m in res}
    assert err[""] < 1.1 * err["element"], err
    bound = 5e-3 if prec == C.PREC_MIXED_HALF else 3e-2
    assert err[""] < bound and np.allclose(res[""][1], norms, rtol=bound, atol=0)


@pytest.mark.parametrize("ls,nrhs", [(6, 1), (12, 3), (20, 2), (8, 1)])
def test_mobius_residual_step_in_last_kernel(monkeypatch, ls, nrhs):
    """Mixed Moebius solves with the residual step in M^dag's last kernel (an
    Ls that does not divide 64) and as a pass of its own (CPS_HIP_R_IN_HOP=0;
    8 always): A p is rounded to FP16 in between only in the second, so the
    residual histories differ in rounding and both meet the FP64 stopping
    rule; the solutions then agree within the tolerance times the condition of
    M^dag M, below 1e4 at this mass."""
    L = [4, 6, 4, 8]
    op = C.make_op(C.OP_MOBIUS, mass=0.1, m5=1.8, b=1.5, c=0.5)
    n = int(np.prod(L)) // 2 * ls
    src = np.concatenate([F.gaussian_fermion(n, 350 + k) for k in range(nrhs)])
    arg = C.make_cg_arg(1e-11, 5000, precision=C.PREC_MIXED_HALF)
    lat = C.Lattice(L, ls, (0, 0, 0, 1))
    lat.import_gauge(wilson_gauge(L, 0.2, 349))
    sol, its = {}, {}
    for mode in ("1", "0"):
        monkeypatch.setenv("CPS_HIP_R_IN_HOP", mode)
        sol[mode], res = lat.invcg(op, src, arg, nrhs=nrhs)
        its[mode] = [r.iterations for r in res]
        assert max(r.true_res for r in res) <= 1e-11
    assert rel(sol["1"], sol["0"]) < 1e-7
    assert max(abs(a - b) / b for a, b in zip(its["1"], its["0"])) < 0.15, its
    lat.close()
