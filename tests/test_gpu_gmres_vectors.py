"""GMRES's vector kernels (csrc/hip/blas.hip): iterates after a set number of
steps against the minimal-residual combination of a Krylov basis that torch
builds from the same product.

The iterate does not depend on how the basis is made, so the two differ by
rounding alone: below 20 steps of products that agree to 1e-14, a second-kind
operator (condition number below 100) and residuals that stay above 1e-6 of
the right-hand side bound it by 20 * 1e-14 * 100 * a few < 1e-10."""
import pytest
import torch

import fmbem_gpu_c_amd as F
from conftest import wavenumber

pytestmark = pytest.mark.gpu


def _best(plan, b, steps):
    """argmin |b - A x| over the Krylov space of b, one right-hand side."""
    V, W = [b / torch.linalg.norm(b)], []
    for _ in range(steps):
        w = plan.matvec(V[-1][None])[0]
        W.append(w)
        v = w.clone()
        for _ in range(2):
            for u in V:
                v = v - torch.vdot(u, v) * u
        V.append(v / torch.linalg.norm(v))
    B, AB = torch.stack(V[:steps], 1), torch.stack(W, 1)
    y = torch.linalg.lstsq(AB.cpu(), b[:, None].cpu()).solution.to(b.device)
    return (B @ y)[:, 0], float(torch.linalg.norm(b - (AB @ y)[:, 0]) / torch.linalg.norm(b))


# one block a vector; a remainder of a block; more elements than an inner product's 128 x 256
# threads and not a multiple of them
@pytest.mark.parametrize("nu,nrhs,steps,restart", [(3, 1, 1, 1), (3, 3, 5, 30), (5, 2, 9, 30),
                                                   (8, 1, 12, 12), (8, 4, 6, 30),
                                                   (43, 2, 4, 30)])
def test_iterates(nu, nrhs, steps, restart):
    m = F.Mesh.ellipsoid(nu, 0.1, 0.09, 0.08, seed=nu)
    t = F.Tree(m)
    plan = F.Plan(t, wavenumber(1000.0), nrhs_max=nrhs)
    g = torch.Generator().manual_seed(nu)
    b = torch.randn((nrhs, t.n), dtype=torch.complex128, generator=g).cuda()
    x, info = plan.gmres(b, restart=restart, tol=1e-14, maxit=steps, check=False)
    assert info.iters == steps
    for r in range(nrhs):
        ref, res = _best(plan, b[r], steps)
        err = float(torch.linalg.norm(x[r] - ref) / torch.linalg.norm(ref))
        print("nu", nu, "rhs", r, "err %.1e residual %.1e" % (err, res), flush=True)
        assert res > 1e-6 and err < 1e-10
        assert abs(info.relres[r] - res) < 1e-10
