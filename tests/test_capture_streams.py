"""A product under the caller's own stream capture stays on the captured
stream: the plan's second stream, which a plain pass of four levels and more
uses, is not forked there (csrc/host/plan.c compiled against recorders)."""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.mark.parametrize("depth", [4, 5, 7])
@pytest.mark.parametrize("transposed", [0, 1])
def test_captured_pass_keeps_to_its_stream(depth, transposed, tmp_path):
    exe = str(tmp_path / "streams")
    subprocess.run(["gcc", "-std=gnu11", "-O1", "-w", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "capture_streams.c"), "-o", exe, "-lm",
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    p = subprocess.run([exe, str(depth), str(transposed)], capture_output=True, text=True,
                       timeout=60)
    plain, captured = [int(v) for v in p.stdout.split()]
    assert plain > 0 and captured == 0, (p.stdout, p.stderr)
