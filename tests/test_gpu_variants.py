"""Launch variants: what the tuner may choose from, and what can be named."""
import ctypes as C
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def make(ns, nx, ny, fp32, members):
    closure = importlib.import_module(ns.__name__ + ".closure")
    L = ns.load()
    h = L.nsd_create_batch(nx, ny, closure.TWO_PI, closure.TWO_PI,
                           ns.NSD_FP32 if fp32 else ns.NSD_FP64, members, None, 0)
    rate = 1e-3 if min(nx, ny) >= 32 else 0.0
    p = closure.params(max(nx, ny), dict(closure.PHYSICS, rate=rate))
    assert L.nsd_set_params(h, C.byref(p)) == 0
    return L, h


def variants(L, h):
    r, c = C.c_int(-1), C.c_int(-1)
    assert L.nsd_get_variants(h, C.byref(r), C.byref(c)) == 0
    return r.value, c.value


def steps(ns, L, h, nx, ny, members, first=1):
    """Last member's field after four steps."""
    seeds = (C.c_ulonglong * members)(*range(first, first + members))
    assert L.nsd_set_member_params(h, None, seeds) == 0
    assert L.nsd_batch_random_phase(h, seeds, 4.0, 1.0) == 0
    assert L.nsd_set_time(h, 0.0, 0.0) == 0 and L.nsd_set_forcing_counter(h, 0) == 0
    assert L.nsd_advance_graph(h, 4, 1) == 0
    w = np.zeros((ny, nx // 2 + 1), np.complex128)
    assert L.nsd_member_download(h, members - 1, w.ctypes.data_as(ns.c_double_p)) == 0
    assert np.linalg.norm(w) > 0
    return w


GRIDS = [(16, 16, False, 3), (32, 32, True, 3), (64, 64, True, 40), (64, 64, False, 300),
         (128, 128, True, 16), (128, 128, False, 90), (256, 256, True, 16), (256, 256, True, 1),
         (256, 512, False, 2), (512, 512, True, 3), (512, 512, True, 9), (1024, 64, True, 2),
         (1024, 1024, True, 2), (1024, 1024, False, 3), (2048, 1024, False, 1)]


@pytest.mark.parametrize("nx,ny,fp32,members", GRIDS)
def test_tuned_launches_keep_the_bits(ns, nx, ny, fp32, members):
    L, h = make(ns, nx, ny, fp32, members)
    start = variants(L, h)
    ref = steps(ns, L, h, nx, ny, members)
    for again in range(2):
        r, c = C.c_int(-1), C.c_int(-1)
        assert L.nsd_autotune(h, 3, 1, C.byref(r), C.byref(c)) == 0
        print(f"{nx} x {ny} x {members} {'FP32' if fp32 else 'FP64'}: starts with {start}, "
              f"tuned {(r.value, c.value)}", flush=True)
        assert variants(L, h) == (r.value, c.value)
        assert np.array_equal(steps(ns, L, h, nx, ny, members), ref)
    # back to the starting ones, whichever they are
    assert L.nsd_set_variants(h, *start) == 0 and variants(L, h) == start
    assert np.array_equal(steps(ns, L, h, nx, ny, members), ref)
    assert L.nsd_set_variants(h, 0, 5) != 0 and L.nsd_set_variants(h, -1, 0) != 0
    assert variants(L, h) == start
    L.nsd_destroy(h)


# variant 0's code in other workgroups
@pytest.mark.parametrize("nx,ny,fp32,members", [
    (16, 32, True, 3), (16, 16, False, 3), (64, 128, True, 5), (64, 64, False, 5),
    (256, 512, True, 2), (512, 256, False, 3), (512, 512, True, 1), (1024, 1024, True, 1),
    (1024, 512, False, 1)])
def test_workgroup_sizes_give_the_same_bits(ns, nx, ny, fp32, members):
    L, h = make(ns, nx, ny, fp32, members)
    assert L.nsd_set_variants(h, 0, 0) == 0
    ref, tried = steps(ns, L, h, nx, ny, members), 0
    for v in (1, 4, 2) if fp32 else (1, 4):
        for pair in ((v, 0), (0, v)):
            if L.nsd_set_variants(h, *pair) == 0:
                tried += 1
                assert np.array_equal(steps(ns, L, h, nx, ny, members), ref), pair
    assert tried >= 2
    L.nsd_destroy(h)
