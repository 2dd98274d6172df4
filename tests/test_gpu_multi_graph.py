"""The graph of several batch contexts is captured again when a call's arguments
change; the replays of the one before it have to end first."""
import ctypes as C
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(64, 128), (256, 32, 512)])
def test_graph_replaced_under_its_replays(ns, sizes):
    closure = importlib.import_module(ns.__name__ + ".closure")
    L, members, out = ns.load(), 3, []
    for wait in (False, True):
        cs = []
        for n in sizes:
            h = L.nsd_create_batch(n, n, closure.TWO_PI, closure.TWO_PI, ns.NSD_FP64, members,
                                   None, 0)
            p = closure.params(n)
            assert L.nsd_set_params(h, C.byref(p)) == 0
            seeds = (C.c_ulonglong * members)(*range(1, members + 1))
            assert L.nsd_set_member_params(h, None, seeds) == 0
            assert L.nsd_batch_random_phase(h, seeds, 4.0, 1.0) == 0
            cs.append(h)
        m = L.nsd_multi_create((C.c_void_p * len(cs))(*cs), len(cs))
        assert m
        for adaptive in (1, 0, 1, 1, 0):  # a fixed step keeps the last adaptive one
            assert L.nsd_multi_advance(m, 20, adaptive) == 0
            if wait:
                assert L.nsd_multi_synchronize(m) == 0
        assert L.nsd_multi_synchronize(m) == 0
        got = []
        for n, h in zip(sizes, cs):
            w = np.zeros((n, n // 2 + 1), np.complex128)
            assert L.nsd_member_download(h, 1, w.ctypes.data_as(ns.c_double_p)) == 0
            got.append(w)
        L.nsd_multi_destroy(m)
        for h in cs:
            L.nsd_destroy(h)
        out.append(got)
    for a, b in zip(*out):
        assert np.linalg.norm(b) > 0 and np.array_equal(a, b)
