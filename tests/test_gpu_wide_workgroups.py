"""The 8-wave form of the translations (csrc/host/rcr.c) against the 4-wave one
that a plan with waves=4 runs, over the orders at which the rule changes (one
and two workgroups a CU, global workspace) and over few and many workgroups,
forward and transposed.

The two add the same products in another order: FP64 2 * 94 * 1.1e-16 per
translation and 189 sources a target, below 1e-13; FP32 the same count of 6e-8
with random signs, below 1e-5."""
import numpy as np
import pytest
import torch

import fmbem_gpu_c_amd as F
from conftest import wavenumber

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tree():
    return F.Tree(F.Mesh.ellipsoid(17, 0.08, 0.07, 0.10, seed=5), depth=5)


@pytest.mark.parametrize("nrhs", [1, 5])
@pytest.mark.parametrize("orders", [[25, 24, 23, 22], [34, 33, 21, 20], [49, 31, 32, 19],
                                    [65, 42, 30, 18], [97, 64, 48, 17]])
def test_eight_waves_match_four(tree, orders, nrhs):
    k = wavenumber(4000.0)
    kw = dict(precision=F.FMB_MIXED, nrhs_max=nrhs, p_rule=F.PRULE_EXPLICIT,
              p_levels=[0, 0] + orders)
    four, rule = F.Plan(tree, k, waves=4, **kw), F.Plan(tree, k, **kw)
    rng = np.random.default_rng(sum(orders))
    x = torch.tensor(rng.standard_normal((nrhs, tree.n)) + 1j * rng.standard_normal((nrhs, tree.n)),
                     device="cuda")
    for prec, tol in ((F.FMB_FP64, 1e-13), (F.FMB_MIXED, 1e-5)):
        for fn in ("matvec_parts", "matvec_t"):
            a = getattr(rule, fn)(x, parts=2, prec=prec)
            b = getattr(four, fn)(x, parts=2, prec=prec)
            e = float(torch.linalg.norm(a - b) / torch.linalg.norm(b))
            print(orders, nrhs, fn, prec, "%.1e" % e, flush=True)
            assert e < tol
