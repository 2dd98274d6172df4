"""The closure's streaming tiles where a workgroup walks several of them, the
evaluation's in-kernel conversion, and an epoch longer than the loss slots."""
import ctypes as C

import numpy as np
import pytest

import closure_oracle as CO
from conftest import rel_l2
from test_gpu_closure import fp, make

pytestmark = pytest.mark.gpu


# 128 x 16: 1024 tiles, two a workgroup on a 256-CU device; 128 x 9: 576, some
# workgroups one and some two; 64 x 1: 16 tiles, most of the device idle
@pytest.mark.parametrize("n,batch", [(64, 1), (128, 9), (128, 16)])
def test_gradient_over_several_tiles(ns, n, batch):
    L, h = make(ns, n, batch, seed=5)
    rng = np.random.default_rng(n + batch)
    P = L.nsd_closure_param_count(h)
    p = (rng.standard_normal(P) * 0.3).astype(np.float32)
    assert L.nsd_closure_params(h, fp(p), 1) == 0
    x = rng.standard_normal((batch, n, n)).astype(np.float32)
    t = rng.standard_normal((batch, n, n)).astype(np.float32)
    g = np.zeros(P, np.float32)
    loss = C.c_double()
    out = g.ctypes.data_as(C.POINTER(C.c_float))
    # twice: the second call finds the first one's gradients in the buffer
    for _ in range(2):
        assert L.nsd_closure_gradient(h, fp(x), fp(t), batch, C.byref(loss), out) == 0
    _, ref = CO.loss_and_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64))
    off = 0
    for ci, co in zip(CO.CIN, CO.COUT):
        nw = co * 9 * ci
        # bf16 operands, as the other gradient tests
        assert rel_l2(g[off:off + nw], ref[off:off + nw]) <= 2e-2
        assert rel_l2(g[off + nw:off + nw + co], ref[off + nw:off + nw + co]) <= 2e-2
        off += nw + co
    L.nsd_closure_destroy(h)


# n = 32: converted by a kernel of its own, from 64 by the input layer; the scale is a
# power of two, so both calls see the same bf16 input
@pytest.mark.parametrize("n,batch", [(32, 2), (64, 3), (128, 5)])
def test_evaluation_converts_its_input(ns, n, batch):
    L, h = make(ns, n, batch)
    rng = np.random.default_rng(n)
    P = L.nsd_closure_param_count(h)
    p = (rng.standard_normal(P) * 0.3).astype(np.float32)
    assert L.nsd_closure_params(h, fp(p), 1) == 0
    x = rng.standard_normal((batch, n, n)).astype(np.float32)
    want = np.zeros_like(x)
    assert L.nsd_closure_forward(h, fp(0.5 * x), batch,
                                 want.ctypes.data_as(C.POINTER(C.c_float))) == 0
    L.nsd_closure_set_scales(h, 0.5, 1.0)
    # device arrays: the data set's own
    assert L.nsd_closure_dataset_reserve(h, batch) == 0
    zero = np.zeros((n, n), np.float32)
    for i in range(batch):
        assert L.nsd_closure_dataset_fill(h, i, fp(x[i]), fp(zero)) == 0
    FP = C.POINTER(C.c_float)
    dx, dy = C.c_void_p(), C.c_void_p()
    assert L.nsd_closure_dataset_slot(h, 0, C.byref(dx), C.byref(dy)) == 0
    a, b = np.zeros_like(x), np.zeros_like(x)

    def evaluate(src, dst):
        assert L.nsd_closure_eval_batch(h, src, dst, batch, None) == 0
        for i in range(batch):
            assert L.nsd_closure_dataset_read(h, i, a[i].ctypes.data_as(FP),
                                              b[i].ctypes.data_as(FP)) == 0

    evaluate(dx, dy)
    assert np.array_equal(a, x) and np.array_equal(b, want)
    evaluate(dx, dx)  # in place
    assert np.array_equal(a, want)
    L.nsd_closure_destroy(h)


def test_epoch_longer_than_the_loss_slots(ns):
    """300 fields, 270 minibatches of one in an epoch, at a learning rate that
    changes no weight: the epoch's loss is the mean of the fields' losses."""
    n, count = 16, 300
    L, h = make(ns, n, 1)
    rng = np.random.default_rng(1)
    xs = rng.standard_normal((count, n, n)).astype(np.float32)
    ts = rng.standard_normal((count, n, n)).astype(np.float32)
    assert L.nsd_closure_dataset_reserve(h, count) == 0
    for i in range(count):
        assert L.nsd_closure_dataset_fill(h, i, fp(xs[i]), fp(ts[i])) == 0
    first, last, valid = C.c_double(), C.c_double(), C.c_double()
    assert L.nsd_closure_train(h, count, 1, 1, 1e-30, 7, C.byref(first), C.byref(last),
                               C.byref(valid)) == 0
    a, b = C.c_double(), C.c_double()
    L.nsd_closure_get_scales(h, C.byref(a), C.byref(b))
    sx, st = np.float32(a.value), np.float32(1) / np.float32(b.value)
    losses = np.zeros(count)
    for i in range(count):
        l = C.c_double()
        assert L.nsd_closure_gradient(h, fp(sx * xs[i]), fp(st * ts[i]), 1, C.byref(l), None) == 0
        losses[i] = l.value
    held = np.arange(count) % 10 == 9
    assert first.value == pytest.approx(losses[~held].mean(), rel=1e-9)
    assert last.value == first.value
    assert valid.value == pytest.approx(losses[held].mean(), rel=1e-9)
    L.nsd_closure_destroy(h)
