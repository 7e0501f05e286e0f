"""Box-major field sums (k_field_box, csrc/hip/field.hip): orders of every
remainder of its four-column groups, counts of right-hand sides on both sides
of its groups of 1, 2 and 4, and points that do not fill a wavefront, against
the oracle's treecode (the same tree, orders and separation in FP64: 1e-10, as
in the other treecode tests)."""
import numpy as np
import pytest
import torch

import fmbem_gpu_c_amd as F
import oracle as O
from conftest import wavenumber

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p2,p3", [(24, 8), (25, 24), (26, 25), (27, 26)])
@pytest.mark.parametrize("nrhs,npts", [(1, 1), (1, 65), (2, 64), (3, 200), (5, 63), (9, 130)])
def test_vs_oracle(p2, p3, nrhs, npts):
    m = F.Mesh.icosphere(3, 0.1)
    V, Fc = m.arrays()
    k, n = wavenumber(4000.0), len(Fc)
    pl = F.Plan(F.Tree(m, depth=3), k, nrhs_max=nrhs, p_rule=F.PRULE_EXPLICIT,
                p_levels=[0, 0, p2, p3])
    ob = O.Bem(V, Fc, k)
    ob.fmm_setup(depth=3, plev={2: p2, 3: p3})
    rng = np.random.default_rng(100 * p2 + nrhs)
    x = rng.standard_normal((nrhs, n)) + 1j * rng.standard_normal((nrhs, n))
    d = rng.standard_normal((npts, 3))
    # also points on the z axis of boxes' frames and beyond the sorted grid
    pts = d / np.linalg.norm(d, axis=1)[:, None] * rng.uniform(0.11, 1.2, npts)[:, None]
    pts[0] = [0.0, 0.0, 5.0]
    got = pl.field(torch.tensor(x, device="cuda"), pts, method="fmm").cpu().numpy()
    want = ob.field(x, pts, fmm=True)
    e = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(p2, p3, nrhs, npts, "%.1e" % e, flush=True)
    assert e < 1e-10


@pytest.mark.parametrize("npts", [1, 3, 4, 5, 63, 257, 4096, 4099])
def test_direct_points_of_a_workgroup(npts):
    """The direct sum takes four points a workgroup with one right-hand side
    and one with more: the same panel sums of 1,280 terms in another order,
    1e-13, off the surface and within the refined rule's distance of it."""
    m = F.Mesh.icosphere(3, 0.1)
    t = F.Tree(m, depth=3)
    k = wavenumber(2000.0)
    rng = np.random.default_rng(npts)
    sig = torch.tensor(rng.standard_normal(t.n) + 1j * rng.standard_normal(t.n), device="cuda")
    pl = F.Plan(t, k, robin=sig, nrhs_max=2)
    x = torch.tensor(rng.standard_normal((2, t.n)) + 1j * rng.standard_normal((2, t.n)),
                     device="cuda")
    d = rng.standard_normal((npts, 3))
    pts = d / np.linalg.norm(d, axis=1)[:, None] * rng.choice([0.101, 0.105, 0.3], npts)[:, None]
    dirs = np.array([[0.0, 0.0, 1.0], [0.6, 0.8, 0.0]])
    both = pl.field(x, pts, dirs)
    for r in range(2):
        one = pl.field(x[r:r + 1].contiguous(), pts, dirs[r:r + 1])
        e = float(torch.linalg.norm(one[0] - both[r]) / torch.linalg.norm(both[r]))
        assert e < 1e-13, (npts, r, e)
