"""The rhs-group mapping of the 4-D hops (several rhs of a site in one
wavefront) at its edges, against the element order: both are forced, without
timing (CPS_HIP_HOP_MODE, CPS_HIP_TUNE=0)."""
import re

import numpy as np
import pytest

import cps_public_amd as C
from cps_public_amd import fields as F
from tests.helpers import rel, wilson_gauge

pytestmark = pytest.mark.gpu

KAPPAS, CSW = [0.130, 0.1325], 1.0
SPATIAL, RHSGROUP = 4, 32   # HopFlags


def _both(monkeypatch, capfd, kind, L, nrhs, precs):
    """{mode: (matpc, matpc^dag, mdagm and norms per precision)}, and the
    flags of every launch in the rhs-group mapping."""
    u = wilson_gauge(L, 0.2, 81)
    n = int(np.prod(L)) // 2
    src = np.concatenate([F.gaussian_fermion(n, 82 + k) for k in range(nrhs)])
    monkeypatch.setenv("CPS_HIP_TUNE", "0")
    monkeypatch.setenv("CPS_HIP_TUNE_REPORT", "1")
    out = {}
    for mode in ("element", "rhsgroup"):
        monkeypatch.setenv("CPS_HIP_HOP_MODE", mode)
        lat = C.Lattice(L, 1, (0, 0, 0, 1))
        lat.import_gauge(u)
        if kind == "clover":
            lat.clover_build(KAPPAS, CSW)
            op = C.make_op(C.OP_CLOVER, mass=1.0 / (2 * KAPPAS[0]) - 4.0, csw=CSW)
        else:
            op = C.make_op(C.OP_WILSON, mass=0.1)
        capfd.readouterr()
        out[mode] = [lat.matpc(op, src, 0, nrhs=nrhs), lat.matpc(op, src, 1, nrhs=nrhs)]
        out[mode] += [lat.mdagm_prec(op, src, p, nrhs=nrhs) for p in precs]
        flags = [int(f) for f in re.findall(r"cps_hip rule: .* flags (\d+)", capfd.readouterr().err)]
        assert flags and all(((f & RHSGROUP) != 0) == (mode == "rhsgroup") for f in flags), flags
        lat.close()
    return out, flags


@pytest.mark.parametrize("kind", ["wilson", "clover"])
@pytest.mark.parametrize("L,nrhs", [([6, 10, 4, 6], 2), ([10, 6, 6, 10], 4), ([6, 4, 6, 10], 6), ([6, 6, 6, 2], 8)])
def test_part_blocks_and_chunks(monkeypatch, capfd, kind, L, nrhs):
    """720, 1800, 720 and 216 sites a parity: the last block of a group of 4
    or 2 rhs and the last 64-site chunk of the partials are parts.  FP64: the
    bits of the element order, |M x|^2 included (same arithmetic, same tree).
    Half precision: separate compilations of one source, so a few elements
    may round to the neighbouring FP16 number (2^-11 of a site's largest
    real): 1e-6 of the whole, and 1e-10 of |M x|^2."""
    out, flags = _both(monkeypatch, capfd, kind, L, nrhs, (C.PREC_DOUBLE, C.PREC_MIXED_HALF))
    e, g = out["element"], out["rhsgroup"]
    assert np.array_equal(e[0], g[0]) and np.array_equal(e[1], g[1])
    assert np.array_equal(e[2][0], g[2][0]) and np.array_equal(e[2][1], g[2][1])
    assert rel(g[3][0], e[3][0]) < 1e-6 and np.max(np.abs(g[3][1] - e[3][1]) / e[3][1]) < 1e-10


@pytest.mark.parametrize("kind", ["wilson", "clover"])
@pytest.mark.parametrize("nrhs", [18, 20])
def test_spatial_sweep_with_part_tile(monkeypatch, capfd, kind, nrhs):
    """16^3x2, FP64: a spatial block holds 256 sites of a slice, so the input
    window (3 slices) of 8 groups of 2 rhs or of 4 groups of 4 fits L2, and
    the 9 and 5 groups of these batches leave a last tile of one.  The bits
    of the element order."""
    out, flags = _both(monkeypatch, capfd, kind, [16, 16, 16, 2], nrhs, (C.PREC_DOUBLE,))
    assert any(f & SPATIAL for f in flags)
    e, g = out["element"], out["rhsgroup"]
    assert np.array_equal(e[0], g[0]) and np.array_equal(e[1], g[1])
    assert np.array_equal(e[2][0], g[2][0]) and np.array_equal(e[2][1], g[2][1])
