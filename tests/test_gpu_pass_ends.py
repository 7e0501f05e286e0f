"""Start and end of a pass (k_begin, k_l2p_near, k_near_t) for the counts of
right-hand sides that their launches split into groups, leaf boxes of more than
a tile's 32 elements and bases of more than a block's 256 coefficients; and the
two-stream order of the levels against the serial one.

A column of a product with several right-hand sides is the product of that
column: the same sums in the same order up to the atomics of the translations,
FP64 1e-13, FP32 1e-5."""
import numpy as np
import pytest
import torch

import fmbem_gpu_c_amd as F
from conftest import wavenumber

pytestmark = pytest.mark.gpu


def _vec(nrhs, n, seed):
    rng = np.random.default_rng(seed)
    return torch.tensor(rng.standard_normal((nrhs, n)) + 1j * rng.standard_normal((nrhs, n)),
                        device="cuda")


def _err(a, b):
    return float(torch.linalg.norm(a - b) / torch.linalg.norm(b))


@pytest.mark.parametrize("depth,p", [(2, 17), (3, 14), (4, 5)])
@pytest.mark.parametrize("nrhs", [2, 3, 4, 5, 8, 9])
def test_columns(depth, p, nrhs):
    t = F.Tree(F.Mesh.ellipsoid(11, 0.08, 0.07, 0.10, seed=2), depth=depth)
    pl = F.Plan(t, wavenumber(1500.0), precision=F.FMB_MIXED, nrhs_max=nrhs,
                p_rule=F.PRULE_EXPLICIT, p_levels=[0, 0] + [p] * (depth - 1))
    x = _vec(nrhs, t.n, nrhs)
    for prec, tol in ((F.FMB_FP64, 1e-13), (F.FMB_MIXED, 1e-5)):
        for fn in ("matvec_parts", "matvec_t"):
            for parts in (1, 2, 3):
                a = getattr(pl, fn)(x, parts=parts, prec=prec)
                b = torch.cat([getattr(pl, fn)(x[r:r + 1].contiguous(), parts=parts, prec=prec)
                               for r in range(nrhs)])
                assert _err(a, b) < tol, (prec, fn, parts)


@pytest.mark.parametrize("depth", [4, 5, 6])
def test_two_streams_match_one(depth):
    t = F.Tree(F.Mesh.ellipsoid(23, 0.08, 0.07, 0.10, seed=3), depth=depth)
    k = wavenumber(3000.0)
    kw = dict(precision=F.FMB_MIXED, nrhs_max=3)
    two, one = F.Plan(t, k, **kw), F.Plan(t, k, serial_levels=1, **kw)
    x = _vec(3, t.n, depth)
    for prec, tol in ((F.FMB_FP64, 1e-13), (F.FMB_MIXED, 1e-5)):
        for fn in ("matvec", "matvec_t"):
            ref = getattr(one, fn)(x, prec=prec)
            for _ in range(3):   # the streams' order of one pass must not matter to the next
                assert _err(getattr(two, fn)(x, prec=prec), ref) < tol, (prec, fn)


@pytest.mark.parametrize("orders", [[16, 14, 11, 9, 6], [20, 16, 15, 12, 14], [5, 5, 17, 5, 4]])
def test_levels_of_one_launch(orders):
    """A pass on one stream runs the finest target-stationary levels, four at
    most, in one launch: five such levels, and levels that end or interrupt
    their run, against a launch a level on two streams."""
    t = F.Tree(F.Mesh.ellipsoid(23, 0.08, 0.07, 0.10, seed=3), depth=6)
    k = wavenumber(3000.0)
    kw = dict(precision=F.FMB_MIXED, nrhs_max=2, p_rule=F.PRULE_EXPLICIT, p_levels=[0, 0] + orders)
    two, one = F.Plan(t, k, **kw), F.Plan(t, k, serial_levels=1, **kw)
    for nrhs in (1, 2):
        x = _vec(nrhs, t.n, nrhs)
        for prec, tol in ((F.FMB_FP64, 1e-13), (F.FMB_MIXED, 1e-5)):
            for fn in ("matvec", "matvec_t"):
                assert _err(getattr(one, fn)(x, prec=prec), getattr(two, fn)(x, prec=prec)) < tol
