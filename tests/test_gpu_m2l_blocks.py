"""Blocks of right-hand sides of the target-stationary M2L (csrc/hip/rcr_ts.hip):
a short last block, whose workgroups end early, beside full ones."""
import pytest
import torch

import fmbem_gpu_c_amd as F
from conftest import wavenumber

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tree():
    return F.Tree(F.Mesh.ellipsoid(23, 0.1, 0.0875, 0.125, seed=3), depth=5)


def _fine_m2l(plan, nrhs, prec):
    """Milliseconds of levels 4 and 5, the best of five."""
    x = torch.randn((nrhs, plan.n), dtype=torch.complex128, device="cuda")
    plan.set_timing(True)
    best = []
    for _ in range(5):
        plan.matvec(x, prec=prec)
        best.append(plan.timing()[1][4:6])
    plan.set_timing(False)
    return sum(min(t) for t in zip(*best))


@pytest.mark.parametrize("prec", [F.FMB_FP64, F.FMB_MIXED])
def test_short_block_costs_less_than_a_full_one(tree, prec):
    """Orders 14: 33 right-hand sides are a block of 32 and one of 1, three
    batches of 16 vectors a pair where 64 take four.  Under 0.85 of the time
    of 64: where the short blocks' workgroups all met the same shader engines,
    the others took as long as for 64 (measured 0.98 to 1.06; 0.63 now)."""
    pl = F.Plan(tree, wavenumber(1500.0), precision=F.FMB_MIXED, nrhs_max=64, serial_levels=1,
                p_rule=F.PRULE_EXPLICIT, p_levels=[0, 0, 16, 14, 14, 14])
    few, full = _fine_m2l(pl, 33, prec), _fine_m2l(pl, 64, prec)
    print("33: %.3f ms, 64: %.3f ms" % (few, full), flush=True)
    assert few < 0.85 * full


def test_half_empty_batches_of_order_16(tree):
    """FP32, order 16: 17 to 29 right-hand sides would leave the second batch of
    a pair's vectors too empty, and level 2 has too few pairs; a plan that holds
    such a count still takes 16 target-stationary.  Both forms are the same
    operator: FP32 1e-6 as in the tests of the kernels (the order of the sums)."""
    kw = dict(precision=F.FMB_MIXED, p_rule=F.PRULE_EXPLICIT, p_levels=[0, 0, 16, 16, 16, 16])
    k = wavenumber(1500.0)
    for nmax in (24, 33):
        pl = F.Plan(tree, k, nrhs_max=nmax, **kw)
        ref = F.Plan(tree, k, nrhs_max=nmax, m2l_tile=255, **kw)
        for nrhs in (1, 15, 16, 17, 24, 29, 30, 33):
            if nrhs > nmax:
                continue
            for l in (2, 3, 4, 5):
                ts = l > 2 and nrhs in (16, 30, 33)
                assert (pl.launch_shape(0, l, nrhs, F.FMB_MIXED)[0] == F.RCR_MODE_TS) == ts
            x = torch.randn((nrhs, pl.n), dtype=torch.complex128, device="cuda")
            a, b = pl.matvec_parts(x, 2, prec=F.FMB_MIXED), ref.matvec_parts(x, 2, prec=F.FMB_MIXED)
            assert float(torch.linalg.norm(a - b) / torch.linalg.norm(b)) < 1e-6, (nmax, nrhs)


@pytest.mark.parametrize("prec", [F.FMB_FP64, F.FMB_MIXED])
@pytest.mark.parametrize("nmax,nrhs", [(3, 3), (40, 5), (33, 33)])
def test_non_finite_column_stays_in_its_column(tree, prec, nmax, nrhs):
    """NaN and infinity in one right-hand side reach no other, in both
    precisions, through a vector a target, several and blocks of them: the other
    columns agree with a pass without it as passes do, FP64 1e-13, FP32 1e-6."""
    pl = F.Plan(tree, wavenumber(1500.0), precision=F.FMB_MIXED, nrhs_max=nmax,
                p_rule=F.PRULE_EXPLICIT, p_levels=[0, 0, 15, 14, 13, 14])
    assert pl.launch_shape(0, 5, nrhs, prec)[0] == F.RCR_MODE_TS
    g = torch.Generator(device="cuda").manual_seed(nrhs)
    x = torch.randn((nrhs, pl.n), dtype=torch.complex128, device="cuda", generator=g)
    want, bad = pl.matvec(x, prec=prec), nrhs // 2
    for v in (float("nan"), float("inf")):
        x[bad, 100] = v
        got = pl.matvec(x, prec=prec)
        keep = [r for r in range(nrhs) if r != bad]
        e = float(torch.linalg.norm(got[keep] - want[keep]) / torch.linalg.norm(want[keep]))
        assert e < (1e-13 if prec == F.FMB_FP64 else 1e-6), (v, e)
        assert not torch.isfinite(got[bad].real).all()
