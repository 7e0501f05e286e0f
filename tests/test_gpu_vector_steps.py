"""GMRES's vector steps (csrc/hip/blas.hip: fmbh_arnoldi, fmbh_resid) by
themselves, without a product beside them: results at the sizes where their
reductions change form, and their time against the bytes that they move."""
import ctypes

import pytest
import torch

import fmbem_gpu_c_amd as F

pytestmark = pytest.mark.gpu


class _Ws(ctypes.Structure):   # fmbh_vecws (csrc/hip/fmb_hip.h)
    _fields_ = [(n, ctypes.c_void_p) for n in ("part", "cnt", "h1", "h2", "nrm", "hp1", "hp2",
                                               "hpn")]


class _Steps:
    def __init__(self, n, nrhs, nv, seed):
        self.L, self.n, self.nrhs, self.nv = ctypes.CDLL(F.LIB_PATH), n, nrhs, nv
        self.L.fmbh_vecws_bytes.restype = ctypes.c_size_t
        self.L.fmbh_vecws_host_bytes.restype = ctypes.c_size_t
        g = torch.Generator(device="cuda").manual_seed(seed)
        self.V = torch.randn((nv + 1, nrhs, n), dtype=torch.complex128, device="cuda", generator=g)
        self.V /= torch.linalg.norm(self.V, dim=2, keepdim=True)
        self.w = torch.randn((nrhs, n), dtype=torch.complex128, device="cuda", generator=g)
        self.dev = torch.empty(self.L.fmbh_vecws_bytes(nv, nrhs, n), dtype=torch.uint8, device="cuda")
        self.host = torch.empty(self.L.fmbh_vecws_host_bytes(nv, nrhs), dtype=torch.uint8,
                                pin_memory=True)
        self.ws = _Ws()
        self.stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert self.L.fmbh_vecws_init(ctypes.byref(self.ws), self._p(self.dev), self._p(self.host),
                                      nv, nrhs, n, self.stream) == 0

    def _p(self, t):
        return ctypes.c_void_p(t.data_ptr())

    def arnoldi(self):
        assert self.L.fmbh_arnoldi(self._p(self.V), self.nv, self._p(self.w), self.nrhs, self.n,
                                   ctypes.byref(self.ws), self.stream) == 0

    def resid(self, b, w, r):
        assert self.L.fmbh_resid(self._p(b), self._p(w), self._p(r), self.nrhs, self.n,
                                 ctypes.byref(self.ws), self.stream) == 0

    def mirror(self):
        """h1, h2 [nv][nrhs] and the norms as the host reads them."""
        torch.cuda.synchronize()
        m = self.nv * self.nrhs
        z = self.host[:32 * m].view(torch.complex128).reshape(2, self.nv, self.nrhs)
        return z[0].clone(), z[1].clone(), self.host[32 * m:].view(torch.float64)[:self.nrhs].clone()


# one element; a block and one more element; one, two and three more blocks than a reduction takes
# in its own launch (64, over vectors or elements); more blocks than threads sum them (256); more
# than an inner product's 128 chunks; more than an update's 2,048
@pytest.mark.parametrize("n,nrhs,nv", [(1, 1, 1), (256, 3, 2), (257, 2, 16), (257, 1, 33),
                                       (64 * 256, 1, 1), (65 * 256, 1, 1), (67280, 2, 3),
                                       (2048 * 256 - 1, 1, 2), (2048 * 256 + 77, 2, 2),
                                       (1000003, 1, 3)])
def test_results(n, nrhs, nv):
    """Sums of n products in FP64, by pieces: at most 30 + n / 32,768 additions
    one after the other, below 64 * 1.1e-16 of the vectors' norms; a subtraction
    of nv vectors adds nv of it.  1e-13."""
    s = _Steps(n, nrhs, nv, n)
    V, w = s.V[:nv].clone(), s.w.clone()
    s.arnoldi()
    h1, h2, nrm = s.mirror()
    norm = torch.linalg.norm(w, dim=1)
    ref1 = torch.stack([torch.stack([torch.vdot(V[j, r], w[r]) for r in range(nrhs)])
                        for j in range(nv)])
    assert ((h1.cuda() - ref1).abs() < 1e-13 * norm).all()
    w1 = w - (ref1[:, :, None] * V).sum(0)
    ref2 = torch.stack([torch.stack([torch.vdot(V[j, r], w1[r]) for r in range(nrhs)])
                        for j in range(nv)])
    assert ((h2.cuda() - ref2).abs() < 1e-13 * nv * norm).all()
    w2 = w1 - (ref2[:, :, None] * V).sum(0)
    tol = 1e-13 * nv * norm
    assert (torch.linalg.norm(s.w - w2, dim=1) < tol).all()
    assert ((nrm.cuda() - torch.linalg.norm(w2, dim=1)).abs() < tol).all()
    if n > nv:
        assert (torch.linalg.norm(s.V[nv] * nrm.cuda()[:, None] - s.w, dim=1) < tol).all()
    b, r = torch.randn_like(w), torch.empty_like(w)
    s.resid(b, w, r)
    ref = torch.linalg.norm(b - w, dim=1)
    assert torch.equal(r, b - w)
    assert ((s.mirror()[2].cuda() - ref).abs() < 1e-13 * ref).all()


def _us(f, reps):
    best = 1e30
    for _ in range(5):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(reps):
            f()
        e1.record()
        e1.synchronize()
        best = min(best, 1e3 * e0.elapsed_time(e1) / reps)
    return best


@pytest.mark.parametrize("n,nrhs,nv", [(10580, 2, 30), (20480, 3, 20), (60500, 64, 15),
                                       (327680, 9, 29)])
def test_time_follows_the_bytes(n, nrhs, nv):
    """A step reads the basis four times.  Under three times these bytes at the
    rate of a copy, and 100 us for its eight launches: with an ordering of the
    whole L2 in every block it was 5 to 22 times as much."""
    a = torch.empty(1 << 27, dtype=torch.float64, device="cuda")
    b = torch.empty_like(a)
    rate = 16.0 * a.numel() / _us(lambda: b.copy_(a), 3)   # bytes a microsecond
    del a, b
    s = _Steps(n, nrhs, nv, 1)
    t, floor = _us(s.arnoldi, 5), 16.0 * n * nrhs * (4 * nv + 7) / rate
    print("n %d nrhs %d nv %d: %.0f us, bytes %.0f us" % (n, nrhs, nv, t, floor), flush=True)
    assert t < 3 * floor + 100
