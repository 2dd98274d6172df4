"""FP32 8192^2 holds the mixed fields in row-pair tiles of pairs and J in 2 x 2 blocks;
the transforms of other fields, the nonlinear term of given spectra and the subgrid
samples of a fine run use the per-field layouts in the same buffers."""
import ctypes as C
import importlib

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def context(ns, n, fp32):
    closure = importlib.import_module(ns.__name__ + ".closure")
    L = ns.load()
    h = L.nsd_create_batch(n, n, closure.TWO_PI, closure.TWO_PI,
                           ns.NSD_FP32 if fp32 else ns.NSD_FP64, 1, None, 0)
    p = closure.params(n, dict(closure.PHYSICS, rate=0.0))
    assert L.nsd_set_params(h, C.byref(p)) == 0
    return L, h


def test_transforms_between_steps_8192_fp32(ns):
    n, D = 8192, ns.c_double_p
    out = []
    nls = []
    for fp32, compat in ((False, True), (True, True), (True, False)):
        print(f"[gpu] fp32 {fp32} compat {compat}", flush=True)
        L, h = context(ns, n, fp32)
        assert L.nsd_state_random_phase(h, 3, 10.0, 1.0) == 0
        w = np.zeros((n, n // 2 + 1), np.complex128)
        if compat:
            assert L.nsd_state_download(h, w.ctypes.data_as(D)) == 0
            k2 = np.fft.fftfreq(n, 1.0 / n)[:, None] ** 2 + np.arange(n // 2 + 1)[None, :] ** 2
            k2[0, 0] = 1.0
            psi, nl = -w / k2, np.zeros_like(w)
            assert L.nsd_nonlinear(h, w.ctypes.data_as(D), psi.ctypes.data_as(D),
                                   nl.ctypes.data_as(D)) == 0
            nls.append(nl)
        if fp32:
            assert L.nsd_advance_graph(h, 2, 1) == 0
            assert L.nsd_state_download(h, w.ctypes.data_as(D)) == 0
            out.append(w)
        L.nsd_destroy(h)
    err = rel_l2(nls[1], nls[0])
    print(f"nonlinear term at 8192^2, FP32 against FP64: rel L2 {err:.2e}", flush=True)
    assert np.linalg.norm(nls[0]) > 0 and err < 1e-5
    assert np.array_equal(*out)


def test_subgrid_sample_of_8192_fp32(ns):
    """From the J that the tiled row stage wrote: both precisions' samples of one
    field.  The coarse grid keeps modes below the field's peak, so the tendency is no
    small difference of two terms that each agree to 1e-5."""
    n, m = 8192, 32
    closure = importlib.import_module(ns.__name__ + ".closure")
    net = closure.Net(m, 1)
    net.reserve(2)
    got = []
    for i, fp32 in enumerate((False, True)):
        print(f"[gpu] fp32 {fp32}", flush=True)
        L, fine = context(ns, n, fp32)
        _, coarse = context(ns, m, fp32)
        assert L.nsd_state_random_phase(fine, 3, 20.0, 1.0) == 0
        x, t = C.c_void_p(), C.c_void_p()
        assert L.nsd_closure_dataset_slot(net.h, i, C.byref(x), C.byref(t)) == 0
        assert L.nsd_subgrid_sample(fine, 0, coarse, x, t) == 0
        a, b = np.zeros((m, m), np.float32), np.zeros((m, m), np.float32)
        F = C.POINTER(C.c_float)
        assert L.nsd_closure_dataset_read(net.h, i, a.ctypes.data_as(F), b.ctypes.data_as(F)) == 0
        got.append((a, b))
        L.nsd_destroy(fine)
        L.nsd_destroy(coarse)
    net.close()
    (x64, t64), (x32, t32) = got
    ex, et = rel_l2(x32, x64), rel_l2(t32, t64)
    print(f"vorticity {ex:.1e}, tendency {et:.1e} of {np.linalg.norm(t64):.2e}", flush=True)
    assert np.linalg.norm(t64) > 0 and ex < 1e-5 and et < 1e-4
