"""The error controller's steps are the plain ones' where it accepts every candidate and
the CFL rule sets dt: the same bits; and its decisions, restored states and step sizes do
not depend on the kernels that a grid starts with."""
import ctypes as C
import importlib

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def run(ns, nx, ny, fp32, scheme, rtol, steps, general=False, rate=0.0):
    closure = importlib.import_module(ns.__name__ + ".closure")
    L = ns.load()
    h = L.nsd_create_batch(nx, ny, closure.TWO_PI, closure.TWO_PI,
                           ns.NSD_FP32 if fp32 else ns.NSD_FP64, 1, None, 0)
    p = closure.params(max(nx, ny), dict(closure.PHYSICS, rate=rate))
    p.scheme = scheme
    if scheme == 0:
        p.hv_on, p.Re = 0, 1e3
    if rtol is not None:
        p.errctl, p.err_rtol, p.err_safety, p.dt_min, p.dt_max = 1, rtol, 0.9, 1e-8, 0.1
    assert L.nsd_set_params(h, C.byref(p)) == 0
    if general:
        assert L.nsd_set_variants(h, 0, 0) == 0
    assert L.nsd_state_random_phase(h, 3, 4.0, 1.0) == 0
    assert L.nsd_set_time(h, 0.0, 0.0) == 0
    assert L.nsd_advance_graph(h, steps, 1) == 0
    w = np.zeros((ny, nx // 2 + 1), np.complex128)
    assert L.nsd_state_download(h, w.ctypes.data_as(ns.c_double_p)) == 0
    t, a, r, e, d = C.c_double(), C.c_ulonglong(), C.c_ulonglong(), C.c_double(), C.c_double()
    assert L.nsd_get_time(h, C.byref(t), None, None) == 0
    if rtol is not None:
        assert L.nsd_errctl_stats(h, 0, C.byref(a), C.byref(r), C.byref(e), C.byref(d)) == 0
    L.nsd_destroy(h)
    return w, t.value, (a.value, r.value), e.value, d.value


@pytest.mark.parametrize("nx,ny,fp32", [
    (16, 16, False), (32, 16, False), (64, 64, False), (128, 512, False), (512, 128, False),
    (256, 256, False), (1024, 1024, False), (2048, 64, False), (64, 64, True), (256, 256, True),
    (512, 512, True), (1024, 1024, True)])
@pytest.mark.parametrize("scheme", [0, 1])
def test_accepted_steps_are_plain_steps(ns, nx, ny, fp32, scheme):
    plain = run(ns, nx, ny, fp32, scheme, None, 4)
    ctl = run(ns, nx, ny, fp32, scheme, 1e6, 4)
    assert ctl[2] == (4, 0)
    assert ctl[1] == plain[1] and np.array_equal(ctl[0], plain[0])


# 2 and more of the first candidates are rejected and restored; field-parallel against
# variant 0, whose sums have another order (FP64 round-off of a difference of 1e-6 to
# 1e-8 of the field, as the runs against the oracle)
@pytest.mark.parametrize("nx,ny,rate", [(16, 16, 0.0), (64, 64, 1e-3), (128, 512, 1e-3),
                                        (512, 256, 0.0), (1024, 1024, 1e-3)])
@pytest.mark.parametrize("scheme", [0, 1])
def test_decisions_do_not_depend_on_the_kernels(ns, nx, ny, rate, scheme):
    a = run(ns, nx, ny, False, scheme, 1e-8, 12, False, rate)
    b = run(ns, nx, ny, False, scheme, 1e-8, 12, True, rate)
    print(f"{nx} x {ny}: {a[2]}, err {a[3]:.4f}, dt {a[4]:.3e}; rel L2 {rel_l2(a[0], b[0]):.1e}",
          flush=True)
    assert a[2] == b[2] and a[2][1] >= 1
    assert a[1] == pytest.approx(b[1], rel=1e-7)
    assert a[3] == pytest.approx(b[3], rel=1e-6) and a[4] == pytest.approx(b[4], rel=1e-6)
    assert rel_l2(a[0], b[0]) <= 1e-9
