"""Products with many vectors (wide.hip) on the GPU: the batched GEMV from 9 vectors and
the experts of a layer from 9 tokens (with more than 72 assignments; split FP4 and IQ3_0 40),
against the CPU oracle. Work items hold 16 vectors and
workgroups 64 weight rows (32 of gate and of up) in 256-column chunks; for large matrices
with many vectors 32 (split FP4: 16), 128 and 128 (256); launches take 4096 assignments. The
sizes lie at the edges of these."""
import ctypes as C

import numpy as np
import pytest
import torch

from objeta_amd import ExpertTable, HipBackend, HipError, MoeExecutor, QGemvShape, QuantBackend, QuantFormat
from objeta_amd.api import check
from oracle import oracle as orc
from test_gpu_grouped import skewed_selection
from test_gpu_moe import FP4, IQ3, Q4, Q5, assert_moe_close, device_table, make_experts, oracle_experts
from test_gpu_qgemv import _assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [QuantFormat.Q4_0, QuantFormat.Q5_0, QuantFormat.IQ3_0])
@pytest.mark.parametrize("rows,cols,batch", [
    (5, 64, 9),        # one short chunk, one ragged row block
    (128, 128, 16),    # exactly one block, one chunk, one vector tile
    (129, 192, 17),    # one row and a half chunk over
    (300, 1216, 33),   # two work items, column ranges with a short last chunk
    (64, 4096, 70),    # eight column ranges, three work items
])
def test_gemv_wide(backend, fmt, rows, cols, batch):
    m = orc.gauss(rows * cols, 60 + rows, 0.02)
    q = orc.quantize_matrix(int(fmt), m, rows, cols)
    xs = orc.gauss(batch * cols, 61 + cols, 1.0)
    dy = backend.alloc(batch * rows * 4)
    QuantBackend(backend).launch_kernel(fmt, None, backend.to_device(q), backend.to_device(xs), dy,
                                        QGemvShape.new(fmt, rows, cols), batch=batch)
    y = dy.download(np.float32, batch * rows).reshape(batch, rows)
    for t in range(batch):
        xt = xs[t * cols:(t + 1) * cols]
        _assert_close(y[t], orc.gemv(int(fmt), q, xt, rows, cols), q, xt, fmt, rows, cols)


def test_gemv_wide_slices(backend):
    """2^20 columns: launches of 64 vectors, 70 in two."""
    test_gemv_wide(backend, QuantFormat.Q4_0, 3, 1 << 20, 70)


def test_gemv_workspace_of_climbing_batches():
    """Batches that climb call by call: the workspace and what it replaced stay within four
    times the largest call's split vectors (64 MiB here)."""
    be = HipBackend(0, 1)
    rows, cols, step, most = 64, 4096, 128, 4096
    q = be.to_device(orc.quantize_matrix(0, orc.gauss(rows * cols, 3, 0.02), rows, cols))
    x, y = be.alloc(4 * most * cols), be.alloc(4 * most * rows)
    quant = QuantBackend(be)
    free = torch.cuda.mem_get_info()[0]
    for batch in range(step, most + 1, step):
        quant.launch_kernel(QuantFormat.Q4_0, None, q, x, y, QGemvShape.new(QuantFormat.Q4_0, rows, cols), batch=batch)
    be.synchronize()
    assert free - torch.cuda.mem_get_info()[0] <= 4 * (4 * most * cols)
    be.close()


@pytest.mark.parametrize("fmt,cols", [(QuantFormat.Q4_0, 4096), (QuantFormat.Q5_0, 4160), (QuantFormat.IQ3_0, 4096)])
def test_gemv_wide_large_matrix(backend, fmt, cols):
    """8260 rows: the large work, the last row block 68 rows deep, a second work item of one
    vector, and (4160 columns) a short last chunk."""
    rows, batch = 8260, 33
    q = orc.quantize_matrix(int(fmt), orc.gauss(rows * cols, 90, 0.02), rows, cols)
    xs = orc.gauss(batch * cols, 91, 1.0)
    dy = backend.alloc(batch * rows * 4)
    QuantBackend(backend).launch_kernel(fmt, None, backend.to_device(q), backend.to_device(xs), dy,
                                        QGemvShape.new(fmt, rows, cols), batch=batch)
    y = dy.download(np.float32, batch * rows).reshape(batch, rows)
    for t in (0, 15, 16, 31, 32):
        xt = xs[t * cols:(t + 1) * cols]
        _assert_close(y[t], orc.gemv(int(fmt), q, xt, rows, cols), q, xt, fmt, rows, cols)


@pytest.mark.parametrize("rows,cols,batch", [
    (5, 128, 9), (128, 256, 16), (300, 1152, 33),
    (8260, 4096, 17), (8260, 4096, 33),  # the large work: a second and a third work item of one vector
    (8260, 4224, 33),                    # with a short last chunk
])
def test_fp4_split_gemv_wide(backend, rows, cols, batch):
    rng = np.random.default_rng(rows + cols)
    w = rng.integers(0, 256, size=rows * cols // 2, dtype=np.uint8)
    s = rng.integers(112, 132, size=rows * cols // 32, dtype=np.uint8)
    xs = orc.gauss(batch * cols, 6, 1.0)
    dy = backend.alloc(batch * rows * 4)
    QuantBackend(backend).launch_kernel_split_fp4(None, backend.to_device(w), backend.to_device(s),
                                                  backend.to_device(xs), dy, rows, cols, batch=batch)
    y = dy.download(np.float32, batch * rows).reshape(batch, rows)
    for t in range(batch):
        ref = orc.fp4_split_gemv(w, s, xs[t * cols:(t + 1) * cols], rows, cols)
        assert float(np.max(np.abs(y[t] - ref))) <= 1e-4 * float(np.max(np.abs(ref)))


def test_gemv_wide_non_finite_and_extreme_vectors(backend):
    """A vector's infinity or NaN stays in that vector's results, its other elements keep
    their scale; vectors of very large and very small magnitude keep full precision."""
    fmt, rows, cols, batch = QuantFormat.Q4_0, 140, 256, 12
    q = orc.quantize_matrix(0, orc.gauss(rows * cols, 7, 0.02), rows, cols)
    xs = orc.gauss(batch * cols, 8, 1.0).reshape(batch, cols).copy()
    xs[1, 3] = np.inf
    xs[2] *= np.float32(1e5)
    xs[2, 200] = -np.inf
    xs[5, 17] = np.nan
    xs[7] *= np.float32(2.0 ** 118)
    xs[8] *= np.float32(2.0 ** -110)
    dy = backend.alloc(batch * rows * 4)
    QuantBackend(backend).launch_kernel(fmt, None, backend.to_device(q), backend.to_device(xs.ravel()), dy,
                                        QGemvShape.new(fmt, rows, cols), batch=batch)
    y = dy.download(np.float32, batch * rows).reshape(batch, rows)
    for t in range(batch):
        ref = orc.gemv(0, q, xs[t], rows, cols)
        if t in (1, 2, 5):
            assert np.array_equal(y[t], ref, equal_nan=True), t
        else:
            assert np.all(np.isfinite(y[t])), t
            assert float(np.max(np.abs(y[t] - ref))) <= 1e-5 * float(np.max(np.abs(ref))), t


@pytest.mark.parametrize("fmt,E,K,T,H,I,shared", [
    (Q4, 16, 4, 9, 256, 128, False),      # few assignments: sets of eight in the direct call
    (Q4, 16, 9, 9, 256, 128, False),      # the smallest batch of 9 tokens that is not few
    (Q5, 3, 2, 33, 192, 64, True),        # short chunks, inter of one row block
    (IQ3, 7, 3, 70, 320, 192, True),
    (FP4, 5, 4, 65, 256, 384, True),
    (Q4, 6, 4, 1030, 64, 64, True),       # two launches' worth of assignments
    (Q4, 2, 2, 33, 1024, 1024, False),    # few assignments again: 66
    (Q4, 2, 2, 65, 1024, 1024, False),    # the large work: two vector tiles, twice, and one over
    (Q4, 2, 2, 37, 1024, 1024, False),    # 74
    (Q5, 2, 1, 47, 1088, 1024, True),     # with a short chunk
    (IQ3, 2, 2, 70, 1024, 1088, False),   # with ragged row blocks
    (FP4, 2, 2, 40, 1152, 1024, True),
])
def test_layer_wide(backend, fmt, E, K, T, H, I, shared):
    """objeta_hip_moe_layer_shared_device at batches, and the direct grouped call on its
    selection where that takes it: the oracle's routing and selected_moe for tokens across
    the batch, and the per-assignment path for all."""
    experts = make_experts(fmt, E + 1, H, I, H, seed=140 + fmt, gen="gauss")
    table, keep = device_table(backend, fmt, experts[:E])
    sh, keep_s = device_table(backend, fmt, experts[E:]) if shared else (None, None)
    w_r = orc.gauss(E * H, 150 + fmt, 0.02)
    xs = orc.gauss(T * H, 160 + fmt, 1.0).reshape(T, H)
    d_x = backend.to_device(xs.ravel())
    d_out, d_ref, d_grp = (backend.alloc(4 * T * H) for _ in range(3))
    d_ids, d_w = backend.alloc(4 * T * K), backend.alloc(4 * T * K)
    moe = MoeExecutor(backend)
    moe.layer_device(fmt, table, backend.to_device(w_r), None, K, T, d_x, d_x, d_out, d_ids, d_w, H, I, H, shared=sh)
    direct = not shared and T * K <= 1024
    if direct:
        moe.grouped_device(fmt, table, d_ids, d_w, T, K, d_x, d_x, d_grp, H, I, H)
    moe.selected_device(fmt, table, d_ids, d_w, T, K, d_x, d_x, d_ref, H, I, H, shared=sh)
    backend.synchronize()
    assert moe.device_error() == 0
    ids = d_ids.download(np.uint32, T * K).reshape(T, K)
    outs = [b.download(np.float32, T * H).reshape(T, H) for b in ([d_out, d_grp] if direct else [d_out])]
    per = d_ref.download(np.float32, T * H).reshape(T, H)
    oe = oracle_experts(fmt, experts)
    for t in {0, 1, T // 3, T // 2, T // 2 + 1, T - 1}:
        rid, rw, _, _ = orc.router(w_r, xs[t], E, H, K, renormalize=True)
        assert np.array_equal(ids[t], rid), t
        sel = [(int(i), float(v)) for i, v in zip(rid, rw)]
        ref = orc.selected_moe(fmt, oe[:E], sel, xs[t], H, I, H, shared=oe[E] if shared else None)
        for out in outs:
            assert_moe_close(out[t] - xs[t], ref)
    for out in outs:
        assert float(np.max(np.abs(out - per))) <= 1e-4 * float(np.max(np.abs(per)))
    del keep, keep_s


def test_layer_wide_output_over_its_input(backend):
    """Past one launch's 4096 assignments with outputs that run over the inputs: out == x with
    wider rows, and with rows as wide, equal the call with buffers of their own."""
    fmt, E, K, T, H, I = Q4, 8, 8, 600, 64, 64
    moe = MoeExecutor(backend)
    d_wr = backend.to_device(orc.gauss(E * H, 5, 0.02))
    xs = orc.gauss(T * H, 6, 1.0)
    d_ids, d_w = backend.alloc(4 * T * K), backend.alloc(4 * T * K)
    for O in (128, 64):
        experts = make_experts(fmt, E, H, I, O, seed=21, gen="gauss")
        table, keep = device_table(backend, fmt, experts)
        d_x, d_out, d_both = backend.to_device(xs), backend.alloc(4 * T * O), backend.alloc(4 * T * O)
        d_both.upload(np.concatenate([xs, np.zeros(T * (O - H), np.float32)]))
        for x, out in ((d_x, d_out), (d_both, d_both)):
            moe.layer_device(fmt, table, d_wr, None, K, T, x, None, out, d_ids, d_w, H, I, O)
        backend.synchronize()
        assert moe.device_error() == 0
        ref = d_out.download(np.float32, T * O)
        assert float(np.max(np.abs(d_both.download(np.float32, T * O) - ref))) <= 1e-4 * float(np.max(np.abs(ref)))
        del keep


def test_layer_past_the_index_range_is_refused():
    """tokens * k * intermediate above 2^31: InvalidInput, whichever kernels a layer's batch
    takes."""
    be = HipBackend(0, 1)
    E, K, T, H, I = 32, 32, 4096, 64, 16448
    one = make_experts(Q4, 1, H, I, H, seed=2, gen="gauss")
    _, keep = device_table(be, Q4, one)
    table = ExpertTable(be, [tuple(keep)] * E)
    d_x, d_wr = be.to_device(orc.gauss(T * H, 1, 1.0)), be.to_device(orc.gauss(E * H, 2, 0.02))
    d_out, d_ids, d_w = be.alloc(4 * T * H), be.alloc(4 * T * K), be.alloc(4 * T * K)
    with pytest.raises(HipError) as e:
        MoeExecutor(be).layer_device(Q4, table, d_wr, None, K, T, d_x, None, d_out, d_ids, d_w, H, I, H)
    assert e.value.kind == "InvalidInput"
    be.synchronize()
    be.close()


def test_wide_out_of_table_and_repeated_experts(backend):
    fmt, E, K, T, H, I, O = Q4, 4, 2, 40, 256, 128, 264
    experts = make_experts(fmt, E, H, I, O, seed=15, gen="gauss")
    sel = skewed_selection(T, K, E, seed=4)
    sel[3] = [(E + 1, 0.5), (0, 0.5)]
    sel[7] = [(1, 0.6), (1, 0.4)]
    xs = orc.gauss(T * H, 1, 1.0).reshape(T, H)
    moe = MoeExecutor(backend)
    table, keep = device_table(backend, fmt, experts)
    ids = np.array([[s[0] for s in row] for row in sel], np.uint32).ravel()
    ws = np.array([[s[1] for s in row] for row in sel], np.float32).ravel()
    out = backend.alloc(4 * T * O)
    moe.grouped_device(fmt, table, backend.to_device(ids), backend.to_device(ws), T, K, backend.to_device(xs.ravel()),
                       None, out, H, I, O)
    backend.synchronize()
    assert moe.device_error() & 1
    got = out.download(np.float32, T * O).reshape(T, O)
    oe = oracle_experts(fmt, experts)
    for t in range(T):
        if t == 3:
            assert np.all(np.isnan(got[t]))
        else:
            assert_moe_close(got[t], orc.selected_moe(fmt, oe, sel[t], xs[t], H, I, O))
    del keep


def test_layer_wide_graph_replays(backend):
    """A captured 48-token layer replayed with eager calls of other sizes on the same
    stream in between: every replay equals the eager call bit for bit."""
    E, K, H, I, T = 16, 4, 1024, 256, 48
    experts = make_experts(Q4, E, H, I, H, seed=171, gen="gauss")
    table, keep = device_table(backend, Q4, experts)
    d_wr = backend.to_device(orc.gauss(E * H, 172, 0.02))
    d_x = backend.to_device(orc.gauss(T * H, 173, 1.0))
    d_out, d_out2 = backend.alloc(4 * T * H), backend.alloc(4 * T * H)
    d_ids, d_w = backend.alloc(4 * T * K), backend.alloc(4 * T * K)
    d_ids2, d_w2 = backend.alloc(4 * T * K), backend.alloc(4 * T * K)
    moe = MoeExecutor(backend)
    st = backend.stream(0)

    def layer(n, out, ids, w):
        moe.layer_device(Q4, table, d_wr, None, K, n, d_x, d_x, out, ids, w, H, I, H, stream=st)

    layer(T, d_out, d_ids, d_w)
    backend.synchronize(st)
    ref = d_out.download(np.float32, T * H)
    check(backend.L.objeta_hip_graph_begin_capture(backend.ctx, st))
    layer(T, d_out, d_ids, d_w)
    g = C.c_void_p()
    check(backend.L.objeta_hip_graph_end_capture(backend.ctx, st, C.byref(g)))
    try:
        for n in (33, 16, 40):
            d_out.upload(np.zeros(T * H, np.float32), st)
            check(backend.L.objeta_hip_graph_launch(backend.ctx, g, st))
            backend.synchronize(st)
            assert np.array_equal(d_out.download(np.float32, T * H), ref), n
            layer(n, d_out2, d_ids2, d_w2)
            backend.synchronize(st)
    finally:
        check(backend.L.objeta_hip_graph_destroy(backend.ctx, g))
    assert moe.device_error() == 0
    del keep
