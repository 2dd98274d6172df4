"""Stage kernels over grid shapes: two steps with FP32 stages against the same
two steps in FP64 on the GPU, which the parity tests hold to the oracle.

Rows and columns of different lengths run different instantiations of the
stage kernels, whose layouts of the mixed fields and of J have to meet.  The
tolerance is FP32 round-off: one step at 4096^2 differs by 7.7e-8 relative L2,
and a layout, a mode or a twiddle that is wrong differs by 1e-3 and more, so
1e-6 bounds two steps."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu
TWO_PI = 2 * np.pi


@pytest.fixture(autouse=True)
def _announce(request):
    print(f"\n[gpu] {request.node.name}", flush=True)


def two_steps(ns, nx, ny, fp32, integrating_factor):
    s = ns.Spectral(nx, ny, TWO_PI, TWO_PI, 1e4)
    s.init(taylor_green=False)
    s.set_precision(fp32)
    s.set_scheme(integrating_factor)
    s.set_drag(0.1)
    s.random_phase(7, k_peak=min(10.0, min(nx, ny) / 12.0))
    s.sync_device()
    assert s.advance_n(2, True) == 0
    assert s.sync_host() == 0
    w, t = s.spec("omega_hat").copy(), s.d.t
    s.close()
    return w, t


# a 4096- or 8192-point side next to another length: the layouts of the square
# grids' stage kernels and J's 2 x 2 blocks are not for them
@pytest.mark.parametrize("nx,ny", [(4096, 64), (64, 4096), (4096, 1024), (1024, 4096),
                                   (8192, 128), (128, 8192), (8192, 4096)])
def test_fp32_rectangles_match_fp64(ns, nx, ny):
    w32, t32 = two_steps(ns, nx, ny, True, True)
    w64, t64 = two_steps(ns, nx, ny, False, True)
    err = rel_l2(w32, w64)
    print(f"{nx} x {ny}: FP32 vs FP64 rel L2 {err:.2e}", flush=True)
    assert err <= 1e-6
    assert t32 == pytest.approx(t64, rel=1e-6)


# 8192 points on sixteen waves, both schemes' column kernels
@pytest.mark.parametrize("integrating_factor", [True, False])
def test_fp32_8192_matches_fp64(ns, integrating_factor):
    w32, t32 = two_steps(ns, 8192, 8192, True, integrating_factor)
    w64, t64 = two_steps(ns, 8192, 8192, False, integrating_factor)
    err = rel_l2(w32, w64)
    print(f"8192^2: FP32 vs FP64 rel L2 {err:.2e}", flush=True)
    assert err <= 1e-6
    assert t32 == pytest.approx(t64, rel=1e-6)
