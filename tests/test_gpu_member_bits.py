"""Members of a batch have the bits of a single run of their grid, precision, Reynolds
number and seed, whatever their number, with the starting launches and with tuned ones."""
import numpy as np
import pytest

from test_gpu_variants import make, steps, variants

pytestmark = pytest.mark.gpu


# FP64 and FP32 of every length that has launch variants, from few waves to several
# per SIMD; 2048 points and more have one launch
@pytest.mark.parametrize("nx,ny,fp32,counts", [
    (16, 16, False, (2, 700)), (32, 32, False, (2, 600)), (64, 64, False, (20, 260)),
    (128, 128, False, (16, 70)), (256, 256, False, (8, 17, 40)), (512, 512, False, (2, 9)),
    (1024, 1024, False, (2, 7)), (2048, 1024, False, (2,)),
    (2048, 2048, False, (2, 6)), (512, 1024, False, (3,)),
    (16, 16, True, (2, 700)), (32, 32, True, (2, 600)), (64, 64, True, (20, 260)),
    (128, 128, True, (16, 70)), (256, 256, True, (8, 17, 40)), (512, 512, True, (2, 5, 24)),
    (1024, 1024, True, (2, 4, 16)), (1024, 512, True, (3, 5)), (2048, 2048, True, (2,))])
def test_members_have_the_bits_of_single_runs(ns, nx, ny, fp32, counts):
    L, h = make(ns, nx, ny, fp32, 1)
    one, start = steps(ns, L, h, nx, ny, 1, first=1000), variants(L, h)
    L.nsd_destroy(h)
    for members in counts:
        L, h = make(ns, nx, ny, fp32, members)
        print(f"{nx} x {ny} x {members}: starts with {variants(L, h)}, one with {start}", flush=True)
        for tune in (False, True):
            if tune:
                assert L.nsd_autotune(h, 3, 0, None, None) == 0
            # the last member's seed is the single run's
            w = steps(ns, L, h, nx, ny, members, first=1001 - members)
            assert np.array_equal(w, one), (members, tune)
        L.nsd_destroy(h)
