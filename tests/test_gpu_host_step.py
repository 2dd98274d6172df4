"""One step on host arrays: the pinned path of small grids against the same step
made of the resident-state calls, whose downloads it replaces."""
import importlib

import numpy as np
import pytest

ns = importlib.import_module("navier-stokes-solvers_amd")
pytestmark = pytest.mark.gpu

SPEC = ("omega_hat", "psi_hat", "u_hat", "v_hat")
PHYS = ("u", "v", "omega")


def _solver(nx, ny, fp32, sfd):
    s = ns.Spectral(nx, ny, 2 * np.pi, 2 * np.pi, 500.0)
    s.init(taylor_green=False)
    s.set_precision(fp32)
    s.d.cfl_factor, s.d.dt = 0.5, 1e-3
    s.random_phase(11, k_peak=min(nx, ny) / 8.0, energy=0.5)
    if sfd:
        s.hv_set(enabled=1, coefficient=1.0, order=4, cutoff_ratio=0.4, sfd_enabled=1,
                 sfd_strength=0.5, sfd_timescale=0.5)
    s.sync_host()
    return s


# 512 x 512 is the largest square grid of the pinned buffer, 1024 x 512 is past it
@pytest.mark.parametrize("nx,ny,fp32,sfd", [
    (16, 16, False, False), (64, 32, False, True), (32, 128, True, True), (128, 128, False, True),
    (256, 256, True, False), (512, 512, False, False), (1024, 512, False, False)])
def test_step_on_host_arrays(nx, ny, fp32, sfd):
    a, b = _solver(nx, ny, fp32, sfd), _solver(nx, ny, fp32, sfd)
    for _ in range(3):
        a.check(a.advance_rk4())
        b.sync_device()
        b.check(b.advance_n(1, False))
        b.check(b.sync_host())
    assert a.d.t == b.d.t and a.d.dt == b.d.dt
    # one rounding of a field of unit size, times the log2(nx ny) <= 19 levels of
    # the transforms on either side
    tol = 40 * (2.0 ** -24 if fp32 else 2.0 ** -53)
    names = SPEC + (("sfd_hat",) if sfd else ())
    for n in names:
        x, y = a.spec(n), b.spec(n)
        assert np.linalg.norm(x - y) <= tol * np.linalg.norm(y), n
    for n in PHYS:
        x, y = a.phys(n), b.phys(n)
        assert np.abs(y).max() > 0
        assert np.linalg.norm(x - y) <= tol * np.linalg.norm(y), n


@pytest.mark.parametrize("nx,ny", [(16, 16), (64, 16), (128, 128), (512, 512)])
def test_reductions_of_host_arrays(nx, ny):
    s = _solver(nx, ny, False, False)
    u, v, w = (s.phys(n) for n in PHYS)
    rng = np.random.default_rng(3)
    u[...], v[...], w[...] = (rng.standard_normal(u.shape) for _ in range(3))
    speed = np.sqrt((u * u + v * v).max())
    dx = 2 * np.pi / max(nx, ny)
    # sums of positive terms: at most one rounding per addition along a tree
    assert s.energy() == pytest.approx(0.5 * (u * u + v * v).mean(), rel=1e-13)
    assert s.enstrophy() == pytest.approx(0.5 * (w * w).mean(), rel=1e-13)
    dt = min(max(min(0.5 * dx / (speed + 1e-12), 0.5 * 500.0 * dx * dx), 1e-8), 0.1)
    assert s.cfl() == pytest.approx(dt, rel=1e-14)
    u[0, 0] = np.inf  # a diverged field gives the smallest step
    assert s.cfl() <= 1e-5
