"""The forcing draw is one workgroup of a row kernel whose size depends on the launch:
its bits must not."""
import ctypes as C
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def draws(ns, n, fp32, kmax, variant, members=1):
    """Coloured state after three steps of fixed dt, of member 0: the scaled draws."""
    closure = importlib.import_module(ns.__name__ + ".closure")
    L = ns.load()
    h = L.nsd_create_batch(n, n, closure.TWO_PI, closure.TWO_PI,
                           ns.NSD_FP32 if fp32 else ns.NSD_FP64, members, None, 0)
    p = closure.params(n, dict(closure.PHYSICS, kmax=kmax))
    p.force_colored, p.force_tau = 1, 0.3
    assert L.nsd_set_params(h, C.byref(p)) == 0
    if variant is not None and L.nsd_set_variants(h, variant, variant) != 0:
        L.nsd_destroy(h)
        return None
    seeds = (C.c_ulonglong * members)(*range(4, 4 + members))
    assert L.nsd_set_member_params(h, None, seeds) == 0
    assert L.nsd_batch_random_phase(h, seeds, 4.0, 1.0) == 0
    assert L.nsd_set_time(h, 0.0, 1e-3) == 0
    assert L.nsd_advance(h, 3, 0) == 0
    A = L.nsd_forcing_modes(h)
    ou = np.zeros(2 * A)
    assert L.nsd_forcing_ou(h, ou.ctypes.data_as(ns.c_double_p), 2 * A, 0) == 0
    L.nsd_destroy(h)
    return ou


# fewer modes than a wave, than the 256 lanes of the sums, and more; drawn in the row
# kernel by one launch and by a kernel of its own by another (128^2, up to 14)
@pytest.mark.parametrize("n,fp32,kmax", [(32, True, 6.0), (64, False, 8.0), (128, True, 9.0),
                                         (128, True, 14.0), (128, False, 40.0),
                                         (512, True, 16.0), (1024, False, 20.0),
                                         (2048, True, 20.0)])
def test_draws_do_not_depend_on_the_launch(ns, n, fp32, kmax):
    ref = draws(ns, n, fp32, kmax, 0)
    assert np.abs(ref).max() > 0
    print(f"{n}^2: {ref.size // 2} modes", flush=True)
    for variant in (None, 1, 2, 3, 4):
        got = draws(ns, n, fp32, kmax, variant)
        assert got is None or np.array_equal(got, ref), variant
    for members in (3, 40) if n < 1024 else (2,):
        assert np.array_equal(draws(ns, n, fp32, kmax, None, members), ref), members
