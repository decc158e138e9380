"""A tuned schedule is taken by cores of the same problem: the grid, the
metric form in use, the CFS-PML layers and the stage fork decide which kernels
a schedule names, so none of them is shared. Each library call runs in a
process of its own, since a process reads the cache file once."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu
REPO = Path(__file__).resolve().parent.parent

CHILD = r"""
import sys
import numpy as np
from cgfd import configs, model
tune, nscen, *probe = sys.argv[1:]
def scenario(kind):
    sc = configs.small(ni=70, nj=52, nk=40, imethod=2, curvilinear=True)
    if kind == "tilted":
        sc.x = (sc.x + 40.0 * np.sin(np.arange(sc.nk) / 9.0)[:, None, None]).astype(np.float32)
    if kind == "layers":
        sc.pml_layers = [[n and n + 1 for n in side] for side in sc.pml_layers]
    return sc
def make(kind):
    st = model.Setup(scenario(kind))
    n = int(nscen)
    return model.Batch(st, [(None, 10)] * n) if n > 1 else model.Core(st)
if tune == "tune":
    c = make("same")
    print(*c.autotune(2)[:2])
for kind in probe:
    c = make(kind)
    if kind == "forked":
        c.set_overlap(True)
        c.set_variant(0)
    print(kind, *c.variant_info())
"""


def _run(cache, *args):
    env = dict(os.environ, CGFD_TUNE_CACHE=str(cache), PYTHONPATH=str(REPO / "gpu-cgfd3d-dynamic_amd"))
    p = subprocess.run([sys.executable, "-c", CHILD, *args], env=env, capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stderr[-2000:]
    return [ln.split() for ln in p.stdout.splitlines()]


@pytest.mark.parametrize("nscen", [1, 2])
def test_tuned_schedule_stays_with_its_problem(built_libs, tmp_path, nscen):
    cache = tmp_path / "tuned"
    (v, z), = _run(cache, "tune", str(nscen))
    # the one-launch form has no slabs and is timed once
    if v in ("32", "33"):
        assert z == "8" and (v == "32" or nscen == 1)
    line = cache.read_text().split()
    cache.write_text(" ".join(line[:-2] + ["24", "16"]) + "\n")
    default = "32" if nscen > 1 else "33"
    got = _run(cache, "look", str(nscen), "same", "tilted", "layers", "forked")
    assert got == [["same", "24", "16"], ["tilted", default, "8"], ["layers", default, "8"], ["forked", default, "8"]]


def test_lines_of_older_files_serve_their_shape(built_libs, tmp_path):
    cache = tmp_path / "tuned"
    # ni nj nk nscen nfault isfree pml variant zchunk
    cache.write_text("70 52 40 1 1 1 31 24 16\n70 52 41 1 1 1 31 20 32\n")
    got = _run(cache, "look", "1", "same", "tilted", "layers")
    assert got == [[k, "24", "16"] for k in ("same", "tilted", "layers")]
