"""Panel bases, near blocks and shape terms (basis.hip, near.hip, shape.hip) at
the edges of their splits over a wavefront: leaf orders around the slot counts
of the tables (16, 32), rules of fewer and more points than a pass of 16 or a
wavefront of 64, and more self-term points than lanes.

The far and near products against the oracle's: both are FP64 evaluations of
the same sums (lengths below 1,000), 1e-9 as in the other oracle tests and
1e-12 for the near field."""
import numpy as np
import pytest
import torch

import fmbem_gpu_c_amd as F
import oracle as O
from conftest import wavenumber

pytestmark = pytest.mark.gpu


def _rand(shape, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


def _robin(n, k):
    return 1j * k * (0.01 + 0.005 * _rand(n, 3))


@pytest.mark.parametrize("p,rule,order,near,nedge", [
    (1, F.RULE_COLLAPSED, 1, 1, 1),      # one point, one slot of the table in use
    (3, F.RULE_COLLAPSED, 4, 3, 22),     # 16 points: the centroid starts a second pass
    (14, F.RULE_GAUSS7, 3, 8, 24),
    (15, F.RULE_COLLAPSED, 5, 9, 30),    # 25 points in two passes, 81 near points, 90 edge points
    (16, F.RULE_COLLAPSED, 2, 8, 21),    # 17 columns: two slots
    (31, F.RULE_GAUSS7, 3, 7, 24),
    (32, F.RULE_GAUSS7, 3, 8, 24),       # 33 columns: one slot
])
def test_products_vs_oracle(p, rule, order, near, nedge):
    m = F.Mesh.icosphere(3, 0.1)
    V, Fc = m.arrays()
    k, n = wavenumber(2000.0), len(Fc)
    sig = _robin(n, k)
    t = F.Tree(m, depth=3)
    pl = F.Plan(t, k, robin=torch.tensor(sig, device="cuda"), p_rule=F.PRULE_EXPLICIT,
                p_levels=[0, 0, p, p], quad_rule=rule, quad_order=order, near_order=near,
                nedge=nedge)
    ob = O.Bem(V, Fc, k, sigma=sig, rule=rule, order=order, nedge=nedge,
               near=(O.RULE_COLLAPSED, near, 2.0))
    ob.fmm_setup(depth=3, plev={2: p, 3: p})
    x = _rand((1, n), 5)
    xt = torch.tensor(x, device="cuda")
    want_near = ob.near_matvec(x)
    want_far = ob.fmm_matvec(x) - want_near
    for part, want, tol in ((1, want_near, 1e-12), (2, want_far, 1e-9)):
        got = pl.matvec_parts(xt, part).cpu().numpy()
        e = np.linalg.norm(got - want) / np.linalg.norm(want)
        print("p", p, "part", part, "%.1e" % e, flush=True)
        assert e < tol


@pytest.mark.parametrize("p,rule,order,near,nedge", [
    (4, F.RULE_COLLAPSED, 1, 1, 1), (15, F.RULE_COLLAPSED, 5, 9, 30), (16, F.RULE_GAUSS7, 3, 8, 24)])
def test_vertex_gradient_sums_over_rhs(p, rule, order, near, nedge):
    """J is a sum over right-hand sides, and so is its gradient: the kernel of
    one right-hand side against that of several.  Central differences of step
    1e-5 of a radius carry rounding of 1e-15 / 1e-5 = 1e-10 and a solve to
    1e-12; 1e-7."""
    m = F.Mesh.icosphere(3, 0.1)
    k = wavenumber(2000.0)
    t = F.Tree(m, depth=3)
    pl = F.Plan(t, k, robin=torch.tensor(_robin(t.n, k), device="cuda"), nrhs_max=3,
                p_rule=F.PRULE_EXPLICIT, p_levels=[0, 0, p, p], quad_rule=rule, quad_order=order,
                near_order=near, nedge=nedge)
    d = np.array([[0.0, 0.0, 1.0], [0.6, 0.0, 0.8], [0.0, -1.0, 0.0]])
    pts = np.random.default_rng(1).uniform(0.15, 0.4, (70, 3))
    x, _ = pl.gmres(pl.rhs_plane_wave(d), tol=1e-12)
    dV = pl.adjoint_grad(x, pts, d, tol=1e-12, vertices=True)[3].cpu().numpy()
    one = sum(pl.adjoint_grad(x[r:r + 1], pts, d[r:r + 1], tol=1e-12, vertices=True)[3].cpu().numpy()
              for r in range(3))
    e = np.linalg.norm(dV - one) / np.linalg.norm(one)
    print("p", p, "gradient %.1e" % e, flush=True)
    assert e < 1e-7
