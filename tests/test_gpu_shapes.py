"""Stage kernels over grid shapes: two steps with FP32 stages against the same
two steps in FP64 on the GPU, which the parity tests hold to the oracle.

Rows and columns of different lengths run different instantiations of the
stage kernels, whose layouts of the mixed fields and of J have to meet.  The
tolerance is FP32 round-off: one step at 4096^2 differs by 7.7e-8 relative L2,
and a layout, a mode or a twiddle that is wrong differs by 1e-3 and more, so
1e-6 bounds two steps."""
import ctypes as C
import importlib

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


# a 2048-, 4096- or 8192-point side next to another length: the layouts of the square
# grids' stage kernels and J's 2 x 2 blocks are not for them
@pytest.mark.parametrize("nx,ny", [(4096, 64), (64, 4096), (4096, 1024), (1024, 4096),
                                   (8192, 128), (128, 8192), (8192, 4096), (2048, 256),
                                   (256, 2048), (2048, 4096)])
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


# The field-parallel kernels, which small launches start with, against variant
# 0: the shortest and longest lines they take, lines of one wave and of several,
# closing passes of radix 2 and 4, workgroups with unused units.  The two
# contract a few products differently (FP64 1e-13, FP32 1e-5 after 10 steps, as
# the launch variants are held to).
@pytest.mark.parametrize("nx,ny", [(16, 16), (32, 16), (64, 64), (128, 32), (256, 512), (512, 64),
                                   (1024, 128), (2048, 256), (16, 1024), (1024, 1024)])
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("kind", ["forced", "sfd"])
def test_field_parallel_kernels_match_variant_0(ns, nx, ny, fp32, kind):
    runs = []
    for variant in (None, 0):
        s = ns.Spectral(nx, ny, TWO_PI, TWO_PI, 1e4 if kind == "forced" else 200.0)
        s.init(taylor_green=False)
        s.set_precision(fp32)
        s.set_scheme(kind == "forced")
        if kind == "forced" and min(nx, ny) >= 32:
            s.set_forcing(4.0, 6.0, 1e-2, seed=3)
        s.random_phase(5, k_peak=min(10.0, min(nx, ny) / 6.0), energy=1.0)
        if kind == "sfd":
            s.hv_set(enabled=1, coefficient=1.0, order=4, cutoff_ratio=0.4, sfd_enabled=1,
                     sfd_strength=0.5, sfd_timescale=1.0)
        if variant is not None:
            assert s.L.nsd_set_variants(s.ctx, variant, variant) == 0
        s.sync_device()
        assert s.advance_n(10, True) == 0
        assert s.sync_host() == 0
        runs.append((s.spec("omega_hat").copy(), s.spec("sfd_hat").copy(), s.d.t))
        s.close()
    (w, f, t), (w0, f0, t0) = runs
    err = rel_l2(w, w0)
    print(f"{nx} x {ny} {'FP32' if fp32 else 'FP64'} {kind}: rel L2 {err:.1e}", flush=True)
    tol = 1e-5 if fp32 else 1e-13
    assert np.linalg.norm(w0) > 0 and err <= tol
    if kind == "sfd":
        assert rel_l2(f, f0) <= tol
    assert t == pytest.approx(t0, rel=1e-6 if fp32 else 1e-13)


# 2048^2 holds the mixed fields in the stage kernels' own layouts (FP32 pairs and J
# in 2 x 2 blocks, FP64 row-pair tiles); the compat transforms, and the nonlinear
# term whose row stage they feed, use the per-field one in the same buffers.
@pytest.mark.parametrize("fp32", [True, False])
def test_layout_transitions_2048(ns, fp32):
    made = []
    for single, compat in ((not fp32, True), (fp32, True), (fp32, False)):
        s = ns.Spectral(2048, 2048, TWO_PI, TWO_PI, 1e4)
        s.init(taylor_green=False)
        s.set_precision(single)
        s.random_phase(3, k_peak=10.0)
        if compat:
            s.L.ns_spectral_compute_velocity_from_vorticity(s.p)
            s.L.ns_spectral_compute_nonlinear_terms(s.p)
            s.check()
        made.append(s)
    other, mine, plain = made
    err = rel_l2(mine.spec("nonlinear_hat"), other.spec("nonlinear_hat"))
    print(f"nonlinear term at 2048^2, FP32 against FP64: rel L2 {err:.2e}", flush=True)
    assert err < 1e-5
    for s in (mine, plain):
        assert s.advance_n(2, True) == 0
        assert s.sync_host() == 0
    assert mine.d.t == plain.d.t
    assert np.array_equal(mine.spec("omega_hat"), plain.spec("omega_hat"))
    for s in made:
        s.close()


# a long call replays several steps at a time; the counts cross that length and its
# multiples, before and after the kernels' arguments changed
@pytest.mark.parametrize("n,fp32,forced", [(64, False, False), (128, True, True), (512, False, True)])
def test_long_calls_are_single_steps(ns, n, fp32, forced):
    def solver():
        s = ns.Spectral(n, n, 2 * np.pi, 2 * np.pi, 1e3)
        s.init(taylor_green=False)
        s.set_precision(fp32)
        s.set_scheme(True)
        s.d.cfl_factor = 0.5
        if forced:
            s.set_forcing(4.0, 6.0, 1e-3, seed=5)
        s.random_phase(9, k_peak=6.0, energy=0.5)
        s.sync_device()
        return s

    def state(s):
        out = np.zeros((s.ny, s.nkx), np.complex128)
        s.check(s.L.nsd_state_download(s.ctx, out.ctypes.data_as(ns.c_double_p)))
        return out

    a, b = solver(), solver()
    for drag, counts in ((0.0, (37, 7, 8, 33)), (0.2, (9, 40))):
        for s in (a, b):
            s.set_drag(drag)
        for k in counts:
            a.check(a.advance_n(k, True))
            for _ in range(k):
                b.check(b.advance_n(1, True))
            assert a.d.t == b.d.t
            assert np.array_equal(state(a), state(b))


# starting variants of batches on either side of the rule's lines, against variant 0:
# FP64 rows and columns of 512 and 1024 points at more than one and more than four
# waves per SIMD, 64 to 256 past one; FP32 the same, with equal bits below 512^2
@pytest.mark.parametrize("n,members,fp32", [
    (1024, 2, False), (1024, 7, False), (512, 5, False), (256, 17, False), (128, 70, False),
    (64, 260, False), (1024, 2, True), (1024, 7, True), (512, 7, True), (512, 13, True),
    (256, 17, True), (128, 70, True), (64, 260, True), (32, 600, True)])
def test_starting_variants_of_batches(ns, n, members, fp32):
    closure = importlib.import_module("navier-stokes-solvers_amd.closure")
    L = ns.load()
    prec = ns.NSD_FP32 if fp32 else ns.NSD_FP64
    picks = (0, members // 2, members - 1)
    out = []
    for general in (False, True):
        h = closure.context(n, prec, members, seeds=range(1, members + 1))
        seeds = (C.c_ulonglong * members)(*range(1, members + 1))
        assert L.nsd_batch_random_phase(h, seeds, 5.0, 1.0) == 0
        if general:
            assert L.nsd_set_variants(h, 0, 0) == 0
        assert L.nsd_advance_graph(h, 5, 1) == 0
        got = np.zeros((len(picks), n, n // 2 + 1), np.complex128)
        for i, m in enumerate(picks):
            assert L.nsd_member_download(h, m, got[i].ctypes.data_as(ns.c_double_p)) == 0
        L.nsd_destroy(h)
        out.append(got)
    if fp32 and n < 512:
        assert np.array_equal(out[0], out[1])
    # five steps of rounding on either side
    assert rel_l2(out[0], out[1]) <= (2e-6 if fp32 else 1e-14)
