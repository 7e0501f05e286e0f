"""A tuned plan keeps the fastest form of every translation, the
target-stationary M2L among them: by the recorded times of the shape cache,
edited here to make either form the faster."""
import json
import os
import subprocess
import sys

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

CHILD = r"""
import json
import numpy as np, torch
import fmbem_gpu_c_amd as F
t = F.Tree(F.Mesh.ellipsoid(17, 0.08, 0.07, 0.10, seed=5), depth=4)
kw = dict(precision=F.FMB_MIXED, nrhs_max=9, p_rule=F.PRULE_EXPLICIT, p_levels=[0, 0, 17, 16, 14])
k = 2 * np.pi * 4000.0 / 343.0
pl, ref = F.Plan(t, k, autotune=1, **kw), F.Plan(t, k, waves=4, **kw)
x = torch.randn((9, t.n), dtype=torch.complex128, device="cuda")
err = [float(torch.linalg.norm(pl.matvec(x, prec=p) - ref.matvec(x, prec=p)) /
             torch.linalg.norm(ref.matvec(x, prec=p))) for p in (F.FMB_FP64, F.FMB_MIXED)]
print(json.dumps({"forms": [list(pl.launch_shape(0, l, 9)) for l in (2, 3, 4)],
                  "tuned": [list(pl.tile_shape_bf(0, l)[:5]) for l in (2, 3, 4)], "err": err}))
"""


def _child(cache):
    p = subprocess.run([sys.executable, "-c", CHILD], cwd=ROOT, capture_output=True, text=True,
                       env=dict(os.environ, FMBEM_TUNE_CACHE=cache), timeout=100)
    assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-2000:]
    d = json.loads(p.stdout.strip().splitlines()[-1])
    assert d["err"][0] < 1e-13 and d["err"][1] < 1e-5   # the order of the sums
    return d


def test_the_faster_form_runs(tmp_path):
    cache = str(tmp_path / "tiles.txt")
    _child(cache)
    lines = [ln.split() for ln in open(cache)]
    ts = [ln for ln in lines if ln[9] == "5"]     # FP64 orders 16 and 14, FP32 order 14
    assert {(ln[2], ln[4]) for ln in ts} >= {("0", "16"), ("0", "14")}
    for ms, target in (("0.0001", True), ("999.0", False)):
        with open(cache, "w") as f:
            for ln in lines:
                f.write(" ".join(ln[:-1] + [ms] if ln[9] == "5" else ln) + "\n")
        d = _child(cache)
        assert len(open(cache).read().splitlines()) == len(lines)   # nothing timed again
        assert d["forms"][0] == d["tuned"][0]                        # order 17: no such form
        for i in (1, 2):
            assert (d["forms"][i][0] == 5) == target, d
            if not target:
                assert d["forms"][i] == d["tuned"][i]
