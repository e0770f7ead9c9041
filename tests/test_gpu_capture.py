"""Calls captured into a graph after an eager call of another size, or of none: what needs no
more workspace than that call made is taken, by whichever kernels have theirs, and every
replay gives the eager result of the same call within the products' bars."""
import ctypes as C

import numpy as np
import pytest

from objeta_amd import ExpertTable, HipBackend, MoeExecutor, QGemvShape, QuantBackend, QuantFormat
from objeta_amd.api import check
from oracle import oracle as orc
from test_gpu_moe import FP4, Q4, Q5, device_table, make_experts
from test_gpu_official import fp4_random_expert, fp8_random_expert, ptr_order

pytestmark = pytest.mark.gpu


@pytest.fixture
def fresh():
    """A context whose streams have no workspaces yet."""
    be = HipBackend(0, 1)
    yield be
    be.close()


def captured_replays(be, st, call, d_out, n, eager_between, replays=3):
    """The outputs of `replays` replays of `call`, with `eager_between` run after each."""
    check(be.L.objeta_hip_graph_begin_capture(be.ctx, st))
    g = C.c_void_p()
    try:
        call()
    finally:
        check(be.L.objeta_hip_graph_end_capture(be.ctx, st, C.byref(g)))
    outs = []
    try:
        for _ in range(replays):
            d_out.upload(np.zeros(n, np.float32), st)
            check(be.L.objeta_hip_graph_launch(be.ctx, g, st))
            be.synchronize(st)
            outs.append(d_out.download(np.float32, n))
            eager_between()
            be.synchronize(st)
    finally:
        check(be.L.objeta_hip_graph_destroy(be.ctx, g))
    return outs


def assert_replays(outs, ref):
    for o in outs:
        assert np.array_equal(o, outs[0])
        assert float(np.max(np.abs(o - ref))) <= 1e-4 * float(np.max(np.abs(ref)))


@pytest.mark.parametrize("rows,cols,before,batch", [
    (200, 512, 0, 16),      # one column range: no workspace of its own on the passes of eight
    (200, 512, 0, 9),
    (300, 2048, 8, 40),     # after a batch of eight
    (300, 2048, 40, 16),    # and smaller ones after a larger
    (300, 2048, 17, 16),
    (33000, 1024, 9, 8),    # the passes after the wide products
])
def test_gemv_captured_after_other_batches(fresh, rows, cols, before, batch):
    be, st, quant = fresh, fresh.stream(0), QuantBackend(fresh)
    q = orc.quantize_matrix(0, orc.gauss(rows * cols, 3, 0.02), rows, cols)
    xs = orc.gauss(batch * cols, 4, 1.0)
    d_q, d_x, d_y = be.to_device(q), be.to_device(xs), be.alloc(4 * max(batch, before) * rows)
    d_xb = be.to_device(orc.gauss(max(before, 1) * cols, 5, 1.0))
    shape = QGemvShape.new(QuantFormat.Q4_0, rows, cols)
    be.synchronize()

    def gemv(x, n):
        quant.launch_kernel(QuantFormat.Q4_0, st, d_q, x, d_y, shape, batch=n)
    if before:
        gemv(d_xb, before)
        be.synchronize(st)
    outs = captured_replays(be, st, lambda: gemv(d_x, batch), d_y, batch * rows,
                            lambda: gemv(d_xb, before) if before else None)
    gemv(d_x, batch)
    be.synchronize(st)
    assert_replays(outs, d_y.download(np.float32, batch * rows))
    ref = orc.gemv(0, q, xs[(batch - 1) * cols:], rows, cols)
    assert float(np.max(np.abs(outs[0][(batch - 1) * rows:] - ref))) <= 1e-4 * float(np.max(np.abs(ref)))


@pytest.mark.parametrize("fmt,E,K,H,I,before,T", [
    (Q5, 8, 8, 2048, 1024, 11, 2),     # 363 MiB of assigned experts, grouped, then 66: per assignment
    (Q4, 8, 4, 256, 128, 16, 3),
    (FP4, 16, 8, 256, 128, 513, 512),  # two launches' worth of assignments, then one
    (Q4, 8, 8, 64, 64, 700, 300),
])
def test_layer_captured_after_other_batches(fresh, fmt, E, K, H, I, before, T):
    be, st, moe = fresh, fresh.stream(0), MoeExecutor(fresh)
    one = make_experts(fmt, 1, H, I, H, seed=9, gen="gauss")
    _, keep = device_table(be, fmt, one)
    table = ExpertTable(be, [tuple(keep)] * E)
    d_wr = be.to_device(orc.gauss(E * H, 11, 0.02))
    most = max(before, T)
    d_x, d_out, d_out2 = be.to_device(orc.gauss(most * H, 12, 1.0)), be.alloc(4 * most * H), be.alloc(4 * most * H)
    d_ids, d_w = be.alloc(4 * most * K), be.alloc(4 * most * K)
    be.synchronize()

    def layer(n, out):
        moe.layer_device(fmt, table, d_wr, None, K, n, d_x, d_x, out, d_ids, d_w, H, I, H, stream=st)
    layer(before, d_out2)
    be.synchronize(st)
    outs = captured_replays(be, st, lambda: layer(T, d_out), d_out, T * H, lambda: layer(before, d_out2))
    layer(T, d_out)
    be.synchronize(st)
    assert moe.device_error() == 0
    assert_replays(outs, d_out.download(np.float32, T * H))


@pytest.mark.parametrize("k,hidden,inter,before,T", [
    (4, 4096, 1408, 5, 1),    # grouped from 257 MiB, then the per-token kernels
    (2, 4096, 1408, 6, 5),
    (8, 256, 128, 600, 300),  # past the grouped path's 4096 assignments, then 2400
    (8, 256, 128, 400, 300),
])
def test_official_layer_captured_after_other_batches(fresh, k, hidden, inter, before, T):
    be, st, moe, n = fresh, fresh.stream(0), MoeExecutor(fresh), 8
    keep = [be.to_device(a) for a in fp4_random_expert(hidden, inter, hidden, 5)]
    sh_keep = [be.to_device(a) for a in fp8_random_expert(hidden, inter, hidden, 6)]
    table, shared = ExpertTable(be, [ptr_order(keep)] * n), ExpertTable(be, [ptr_order(sh_keep)])
    most = max(before, T)
    rng = np.random.default_rng(k)
    ids = np.array([rng.choice(n, k, replace=False) for _ in range(most)], np.uint32)
    d_ids, d_w = be.to_device(ids.ravel()), be.to_device(rng.dirichlet(np.ones(k), most).astype(np.float32).ravel())
    d_x = be.to_device(orc.gauss(most * hidden, 13, 1.0))
    d_out, d_out2 = be.alloc(4 * most * hidden), be.alloc(4 * most * hidden)
    be.synchronize()

    def layer(t, out):
        moe.official_fp4_device(table, d_ids, d_w, t, k, d_x, out, hidden, inter, hidden, 10.0, st, shared)
    layer(before, d_out2)
    be.synchronize(st)
    outs = captured_replays(be, st, lambda: layer(T, d_out), d_out, T * hidden, lambda: layer(before, d_out2))
    layer(T, d_out)
    be.synchronize(st)
    assert moe.device_error() == 0
    ref = d_out.download(np.float32, T * hidden).astype(np.float64)
    for o in outs:
        assert np.array_equal(o, outs[0])
        # the two forms' sums run in other orders, which moves an FP8 code of an intermediate
        # now and then (one step of 2^-3 of one of the `inter` terms of a result)
        assert np.linalg.norm(o - ref) <= 1e-3 * np.linalg.norm(ref)
