"""Target-stationary M2L (csrc/hip/rcr_ts.hip) on the GPU: against the oracle's
FMM on the same tree and orders, and against the offset-batched kernels (which
a plan with another m2l_tile runs) over the orders, right-hand-side counts and
pair counts that it takes.

The kernels differ in summation order only.  A translation's rounding is
bounded by its row lengths (2 p) and a target's by its <= 189 sources:
FP64 (2 * 16 + 189) * 1.1e-16 < 1e-13, FP32 the same count of 6e-8, 1.4e-5,
as a bound on every element; random signs leave the norms well under 1e-6."""
import numpy as np
import pytest
import torch

import fmbem_gpu_c_amd as F
import oracle as O
from conftest import wavenumber

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sphere4():
    m = F.Mesh.icosphere(4, 0.1)
    V, Fc = m.arrays()
    return m, V, Fc, F.Tree(m, depth=5)


@pytest.fixture(scope="module")
def ellipsoid():
    m = F.Mesh.ellipsoid(17, 0.08, 0.07, 0.10, seed=5)
    return m, F.Tree(m, depth=5)


def _rand(shape, seed):
    rng = np.random.default_rng(seed)
    return torch.tensor(rng.standard_normal(shape) + 1j * rng.standard_normal(shape), device="cuda")


def _err(a, b):
    return float(torch.linalg.norm(a - b) / torch.linalg.norm(b))


@pytest.mark.parametrize("orders", [[16, 15, 14, 13], [12, 9, 8, 5], [4, 3, 2, 1]])
def test_matches_oracle(sphere4, orders):
    """Far field, three right-hand sides, orders on both sides of the row
    groups of four: FP64 1e-9, FP32 1e-5 (the tolerances of the other
    translation modes' oracle tests)."""
    m, V, Fc, t = sphere4
    k = wavenumber(3000.0)
    pl = F.Plan(t, k, precision=F.FMB_MIXED, nrhs_max=3, p_rule=F.PRULE_EXPLICIT,
                p_levels=[0, 0] + orders)
    ob = O.Bem(V, Fc, k)
    ob.fmm_setup(depth=5, plev=dict(zip(range(2, 6), orders)))
    x = _rand((3, Fc.shape[0]), 71)
    xh = x.cpu().numpy()
    far = ob.fmm_matvec(xh) - ob.near_matvec(xh)
    for prec, tol in ((F.FMB_FP64, 1e-9), (F.FMB_MIXED, 1e-5)):
        got = pl.matvec_parts(x, 2, prec=prec).cpu().numpy()
        e = np.linalg.norm(got - far) / np.linalg.norm(far)
        print("orders", orders, "prec", prec, "vs oracle %.2e" % e, flush=True)
        assert e < tol


@pytest.mark.parametrize("nrhs_max", [1, 2, 5, 9, 16, 19, 40])
@pytest.mark.parametrize("orders", [[16, 14, 13, 14], [15, 11, 6, 1]])
def test_matches_offset_batched(ellipsoid, nrhs_max, orders):
    """Uneven boxes; as many right-hand sides as the plan holds, one, and a
    count between (the plan's second pair list); forward and transposed."""
    m, t = ellipsoid
    n = t.n
    kw = dict(precision=F.FMB_MIXED, nrhs_max=nrhs_max, p_rule=F.PRULE_EXPLICIT,
              p_levels=[0, 0] + orders)
    k = wavenumber(4000.0)
    a, b = F.Plan(t, k, **kw), F.Plan(t, k, m2l_tile=255, **kw)
    for nrhs in sorted({1, (nrhs_max + 1) // 2, nrhs_max}):
        x = _rand((nrhs, n), 72 + nrhs)
        for prec, tol in ((F.FMB_FP64, 1e-13), (F.FMB_MIXED, 1e-6)):
            e = _err(a.matvec_parts(x, 2, prec=prec), b.matvec_parts(x, 2, prec=prec))
            et = _err(a.matvec_t(x, parts=2, prec=prec), b.matvec_t(x, parts=2, prec=prec))
            assert e < tol and et < tol, (nrhs, prec, e, et)


def test_non_finite_right_hand_side_stays_in_its_vector(ellipsoid):
    """A NaN in one right-hand side reaches no other: absent vectors of a
    batch repeat its first and are summed nowhere."""
    m, t = ellipsoid
    pl = F.Plan(t, wavenumber(4000.0), nrhs_max=3, p_rule=F.PRULE_EXPLICIT,
                p_levels=[0, 0, 16, 14, 13, 14])
    x = _rand((3, t.n), 73)
    want = pl.matvec(x)
    x[1, 100] = float("nan")
    got = pl.matvec(x)
    assert _err(got[0], want[0]) < 1e-13 and _err(got[2], want[2]) < 1e-13
    assert torch.isnan(got[1].real).any()


def test_graph_replays_match_eager(ellipsoid):
    """Two plans captured into one graph and replayed three times, with an
    eager pass between."""
    m, t = ellipsoid
    plans = [F.Plan(t, wavenumber(f), precision=F.FMB_MIXED, nrhs_max=4) for f in (2000.0, 3000.0)]
    x = _rand((8, t.n), 74)
    for prec, tol in ((F.FMB_FP64, 1e-13), (F.FMB_MIXED, 1e-6)):
        want = torch.cat([p.matvec(x[4 * i:4 * i + 4].contiguous(), prec=prec)
                          for i, p in enumerate(plans)])
        got = F.matvec_batch(plans, [4, 4], x, graph=True, prec=prec, reps=3)
        torch.cuda.synchronize()
        for r in range(3):
            assert _err(got[r], want) < tol, (prec, r)
