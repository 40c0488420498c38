"""Host vectors large enough to be staged through the pinned buffers (from 8
chunks of 2 MiB), against the plain copies of single right-hand sides."""
import numpy as np
import pytest

import cps_public_amd as C
from cps_public_amd import fields as F
from tests.helpers import wilson_gauge

pytestmark = pytest.mark.gpu

L, LS = [12, 6, 10, 8], 10
N = 24 * int(np.prod(L)) // 2 * LS   # 5.5 MB: a single rhs is copied plainly


@pytest.mark.parametrize("nrhs", [4, 12])   # 22.1 MB and 66.4 MB, the last chunk a part
def test_staged_vectors_match_single_rhs_calls(nrhs):
    """The copies move bytes, and a rhs's arithmetic does not depend on the
    batch: every rhs of the batched M^dag M has the bits of its own call."""
    op = C.make_op(C.OP_MOBIUS, mass=0.05, m5=1.8, b=1.5, c=0.5)
    lat = C.Lattice(L, LS, (0, 0, 0, 1))
    lat.import_gauge(wilson_gauge(L, 0.2, 77))
    src = np.concatenate([F.gaussian_fermion(N // 24, 78 + k) for k in range(nrhs)])
    assert src.nbytes >= 16 << 20 and src.nbytes % (2 << 20)
    keep = src.copy()
    out, norms = lat.mdagm(op, src, nrhs=nrhs)
    again, _ = lat.mdagm(op, src, nrhs=nrhs)
    assert np.array_equal(src, keep) and np.array_equal(out, again)
    for k in range(nrhs):
        one, nk = lat.mdagm(op, src[k * N:(k + 1) * N], nrhs=1)
        assert np.array_equal(out[k * N:(k + 1) * N], one) and norms[k] == nk[0]
    lat.close()
