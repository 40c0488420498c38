"""The CG residual step in the epilogue of M^dag's last hop (CLOV_NRR), at the
shapes whose launch rule differs from the other hops'."""
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
