"""A run that is interrupted (a transform of another field in between, its state taken
over into a new context) steps on with the bits of a run that was not: the derivative
fields that are formed again from the state are those that the last step left."""
import ctypes as C
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _context(ns, nx, ny, fp32, scheme):
    closure = importlib.import_module(ns.__name__ + ".closure")
    L = ns.load()
    h = L.nsd_create_batch(nx, ny, closure.TWO_PI, closure.TWO_PI,
                           ns.NSD_FP32 if fp32 else ns.NSD_FP64, 1, None, 0)
    p = closure.params(max(nx, ny), dict(closure.PHYSICS, rate=0.0))
    p.scheme = scheme
    if scheme == 0:
        p.hv_on, p.Re = 0, 1e3
    assert L.nsd_set_params(h, C.byref(p)) == 0
    return L, h


def _state(ns, L, h, nx, ny):
    w = np.zeros((ny, nx // 2 + 1), np.complex128)
    assert L.nsd_state_download(h, w.ctypes.data_as(ns.c_double_p)) == 0
    return w


# every length of the field-parallel kernels, the tiled layouts of 2048 points, and the
# small FP32 grids' kernels
@pytest.mark.parametrize("nx,ny,fp32", [
    (16, 16, False), (32, 64, False), (64, 32, False), (128, 128, False), (256, 512, False),
    (1024, 256, False), (512, 1024, False), (1024, 1024, False), (2048, 2048, False),
    (32, 32, True), (128, 128, True), (256, 256, True), (512, 512, True), (1024, 512, True),
    (512, 1024, True), (1024, 1024, True), (2048, 2048, True)])
@pytest.mark.parametrize("scheme", [0, 1])
def test_interrupted_run_keeps_its_bits(ns, nx, ny, fp32, scheme):
    D = ns.c_double_p
    runs = []
    for cut in (None, "transform", "restart"):
        L, h = _context(ns, nx, ny, fp32, scheme)
        assert L.nsd_state_random_phase(h, 3, 4.0, 1.0) == 0
        assert L.nsd_advance_graph(h, 2, 1) == 0
        if cut == "transform":
            f, g = np.ones((ny, nx)), np.zeros((ny, nx // 2 + 1), np.complex128)
            assert L.nsd_physical_to_spectral(h, f.ctypes.data_as(D), g.ctypes.data_as(D)) == 0
        elif cut == "restart":
            w, t, dt = _state(ns, L, h, nx, ny), C.c_double(), C.c_double()
            assert L.nsd_get_time(h, C.byref(t), C.byref(dt), None) == 0
            L.nsd_destroy(h)
            L, h = _context(ns, nx, ny, fp32, scheme)
            assert L.nsd_state_upload(h, w.ctypes.data_as(D)) == 0
            assert L.nsd_set_time(h, t, dt) == 0
        assert L.nsd_advance_graph(h, 3, 1) == 0
        t = C.c_double()
        assert L.nsd_get_time(h, C.byref(t), None, None) == 0
        runs.append((_state(ns, L, h, nx, ny), t.value))
        L.nsd_destroy(h)
    (w, t), *cuts = runs
    assert np.linalg.norm(w) > 0
    for w1, t1 in cuts:
        assert t1 == t and np.array_equal(w1, w)
