"""Stored choices of the launch tuner (NSD_TUNE_FILE), in a process of their own:
the file is read once per process."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

SCRIPT = r"""
import ctypes as C, importlib, sys
import numpy as np
sys.path.insert(0, sys.argv[1])
ns = importlib.import_module("navier-stokes-solvers_amd")
closure = importlib.import_module("navier-stokes-solvers_amd.closure")
L = ns.load()

def run(n, prec, members, tune):
    h = L.nsd_create_batch(n, n, closure.TWO_PI, closure.TWO_PI, prec, members, None, 0)
    p = closure.params(n)
    assert L.nsd_set_params(h, C.byref(p)) == 0
    rv, cv = C.c_int(-1), C.c_int(-1)
    if tune:
        assert L.nsd_autotune(h, 2, 0, C.byref(rv), C.byref(cv)) == 0
    else:
        assert L.nsd_set_variants(h, 0, 0) == 0
    seeds = (C.c_ulonglong * members)(*range(1, members + 1))
    assert L.nsd_set_member_params(h, None, seeds) == 0
    assert L.nsd_batch_random_phase(h, seeds, 5.0, 1.0) == 0
    assert L.nsd_advance_graph(h, 3, 1) == 0
    w = np.zeros((n, n // 2 + 1), np.complex128)
    assert L.nsd_member_download(h, members - 1, w.ctypes.data_as(ns.c_double_p)) == 0
    L.nsd_destroy(h)
    return w, rv.value, cv.value

for n, prec, members in ((256, ns.NSD_FP32, 40), (128, ns.NSD_FP64, 90)):
    w, rv, cv = run(n, prec, members, True)
    ref = run(n, prec, members, False)[0]
    print(n, prec, members, rv, cv, np.linalg.norm(w - ref) / np.linalg.norm(ref), flush=True)
"""


# per grid: (row, column) values that are no variant, or that belong to another grid.
# An entry without the grid is of an older form, whose numbers meant other kernels.
@pytest.mark.parametrize("row,col", [(77, 77), (-1, 5), (3, 3)])
def test_stored_variants_are_checked(ns, tmp_path, row, col):
    f = tmp_path / "tune"
    lines = []
    for n, other, prec, members in ((256, 2048, ns.NSD_FP32, 40), (128, 4096, ns.NSD_FP64, 90)):
        for kind, v in (("row", row), ("col", col)):
            lines.append(f"{kind} {n} {prec} {members} {v}")
            lines.append(f"{kind} {n}x{other} {prec} {members} 0")
            if v != 3 or prec == ns.NSD_FP32:  # FP32 grids below 512^2 keep one rounding
                lines.append(f"{kind} {n}x{n} {prec} {members} {v}")
    f.write_text("\n".join(lines) + "\n")
    out = subprocess.run([sys.executable, "-c", SCRIPT, ROOT], check=True, timeout=100,
                         env=dict(os.environ, NSD_TUNE_FILE=str(f)), stdout=subprocess.PIPE,
                         text=True).stdout
    print(out, flush=True)
    got = [line.split() for line in out.splitlines() if line and line[0].isdigit()]
    assert len(got) == 2
    for n, prec, members, rv, cv, err in got:
        fp32 = int(prec) == ns.NSD_FP32
        for v in (int(rv), int(cv)):
            assert 0 <= v < 5 and not (fp32 and v == 3)
        # three steps of rounding on either side; a launch that did nothing differs by 1
        assert float(err) <= (1e-6 if fp32 else 1e-14)
    # what was timed instead is stored with its grid
    stored = [line.split() for line in f.read_text().splitlines()]
    for kind in ("row", "col"):
        last = [s for s in stored if s[0] == kind and s[1] == "256x256"][-1]
        assert 0 <= int(last[-1]) < 5 and int(last[-1]) != 3
