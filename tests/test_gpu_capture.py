"""Products captured into a graph by the caller (torch.cuda.graph), replayed
with eager products between the replays: the same operator, FP64 1e-13 and
FP32 pass 1e-5 (the order of the target sums)."""
import numpy as np
import pytest
import torch

import fmbem_gpu_c_amd as F
from conftest import wavenumber

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth", [3, 4, 5])
def test_replays(depth):
    t = F.Tree(F.Mesh.ellipsoid(12, 0.08, 0.07, 0.10, seed=3), depth=depth)
    pl = F.Plan(t, wavenumber(4000.0), precision=F.FMB_MIXED, nrhs_max=2)
    rng = np.random.default_rng(depth)
    xs = [torch.tensor(rng.standard_normal((2, t.n)) + 1j * rng.standard_normal((2, t.n)),
                       device="cuda") for _ in range(3)]
    x = xs[0].clone()
    for prec, tol in ((F.FMB_FP64, 1e-13), (F.FMB_MIXED, 1e-5)):
        want = [(pl.matvec(v, prec=prec), pl.matvec_t(v, prec=prec)) for v in xs]
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            y, yt = pl.matvec(x, prec=prec), pl.matvec_t(x, prec=prec)
        for v, (a, at) in zip(xs, want):
            x.copy_(v)
            g.replay()
            torch.cuda.synchronize()
            for got, ref in ((y, a), (yt, at), (pl.matvec(v, prec=prec), a)):
                e = float(torch.linalg.norm(got - ref) / torch.linalg.norm(ref))
                assert e < tol, (depth, prec, e)
