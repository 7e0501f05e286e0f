"""Plan.launch_shape: the form that a pass of so many right-hand sides takes,
which the rule's shape (Plan.tile_shape) alone does not name."""
import pytest
import torch

import fmbem_gpu_c_amd as F
from conftest import wavenumber

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tree():
    return F.Tree(F.Mesh.ellipsoid(17, 0.08, 0.07, 0.10, seed=5), depth=5)


def _plan(tree, orders, **kw):
    return F.Plan(tree, wavenumber(4000.0), precision=F.FMB_MIXED, p_rule=F.PRULE_EXPLICIT,
                  p_levels=[0, 0] + orders, **kw)


def test_target_stationary_levels(tree):
    pl = _plan(tree, [20, 17, 16, 14], nrhs_max=3)
    for l, ts in ((2, False), (3, False), (4, True), (5, True)):
        assert (pl.launch_shape(0, l, 1)[0] == F.RCR_MODE_TS) == ts, l
    assert pl.launch_shape(0, 5, 3) == (F.RCR_MODE_TS, 2, 0, 16, 0)
    # a requested tile order keeps the offset-batched kernel
    old = _plan(tree, [20, 17, 16, 14], nrhs_max=3, m2l_tile=255)
    assert old.launch_shape(0, 5, 3) == (F.RCR_MODE_LDS,) + old.tile_shape_bf(0, 5)[1:5]


def test_eight_wave_forms(tree):
    """FP64 orders whose batches leave room for one workgroup a CU, and the
    global workspace, take 8 waves; so do launches of few workgroups."""
    pl = _plan(tree, [62, 42, 31, 18], nrhs_max=9)
    assert pl.tile_shape(0, 2)[:1] + pl.tile_shape(0, 2)[3:] == (F.RCR_MODE_GWS, 4, 0.0)
    assert pl.launch_shape(0, 2, 9)[3] == 8 and pl.launch_shape(0, 4, 9)[3] == 8
    assert pl.launch_shape(0, 5, 9, F.FMB_MIXED)[3] == 4
    assert pl.launch_shape(1, 3, 1)[3] == 8
    four = _plan(tree, [62, 42, 31, 18], nrhs_max=9, waves=4)
    for l in range(2, 6):
        for nrhs in (1, 9):
            assert four.launch_shape(0, l, nrhs) == four.tile_shape_bf(0, l)[:5]


def test_refusals(tree):
    pl = _plan(tree, [16, 15, 14, 13], nrhs_max=2)
    for args in ((3, 4, 1), (0, 1, 1), (0, 6, 1), (1, 2, 1), (0, 4, 0), (0, 4, 3)):
        with pytest.raises(F.FmbError) as e:
            pl.launch_shape(*args)
        assert e.value.code == -1
    valu = F.Plan(tree, wavenumber(4000.0), rcr_path=F.RCR_VALU)
    assert valu.launch_shape(0, 5, 1) == (0, 0, 0, 0, 0)


def test_passes_on_two_streams_keep_to_four_waves(tree):
    """FP64, several right-hand sides, and most of M2L's work in levels without
    an 8-wave form: the streams hide more with 4 waves in every launch (327,680
    triangles at 10 kHz with nine right-hand sides 326 ms, 341 with 8 waves).
    Not with one right-hand side, on one stream, or with most of the work in
    levels of that form."""
    pairs = [len(tree.pairs(l)[0]) for l in range(2, 6)]

    def share(orders):
        w = [n * p ** 3 for n, p in zip(pairs, orders)]
        return sum(w[:2]) / sum(w)

    few, most = [44, 30, 21, 20], [94, 62, 21, 20]
    assert share(few) < 0.45 and share(most) > 0.55
    pl = _plan(tree, few, nrhs_max=4)
    waves = lambda p, n: [p.launch_shape(0, l, n)[3] for l in range(2, 6)]  # noqa: E731
    assert waves(pl, 1)[:2] == [8, 8] and waves(pl, 4) == [4, 4, 4, 4]
    assert waves(_plan(tree, few, nrhs_max=4, serial_levels=1), 4)[:2] == [8, 8]
    assert waves(_plan(tree, most, nrhs_max=4), 4)[:2] == [8, 8]
    # FP32, whose batches take half the LDS, on either stream count
    assert pl.launch_shape(0, 2, 4, F.FMB_MIXED)[3] == 8
    x = torch.randn((4, pl.n), dtype=torch.complex128, device="cuda")
    ref = _plan(tree, few, nrhs_max=4, serial_levels=1)
    for fn in ("matvec", "matvec_t"):
        a, b = getattr(pl, fn)(x), getattr(ref, fn)(x)
        assert float(torch.linalg.norm(a - b) / torch.linalg.norm(b)) < 1e-13   # order of the sums
