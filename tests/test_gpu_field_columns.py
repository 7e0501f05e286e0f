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
