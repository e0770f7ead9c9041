"""The framework's work in the sizes it is used at, for timing and for checking.

Each case is a dict of plain values. `prepare` makes what a program holds before the
call (weights, expert tables, activations, captured graphs), `run` makes one pass
through a public entry point, `exact` computes the same outputs in 64 bits with plain
torch, `work` counts the bytes and operations of a pass, `tolerance` states how far a
correct result may lie from another.

Kinds: gemv (QuantBackend.launch_kernel / launch_kernel_split_fp4), layer
(MoeExecutor.layer_device), stack (a decode step of several layers replayed from a
graph), official (MoeExecutor.official_fp4_device), executor
(MoeExecutor.execute_selected_moe_cuda, host in and host out), quantize (the device
quantizer).
"""
from __future__ import annotations

import ctypes as C
import functools
import math

import numpy as np
import torch

from objeta_amd import (ExpertCache, ExpertTable, HipBackend, MoeExecutor, QGemvShape, QuantBackend, QuantFormat,
                        check)
from objeta_amd.api import HostExpertSet

FORMATS = {"q4_0": QuantFormat.Q4_0, "q5_0": QuantFormat.Q5_0, "iq3_0": QuantFormat.IQ3_0,
           "fp4": QuantFormat.DeepSeekFp4E2M1}
BLOCK_BYTES = {"q4_0": 18, "q5_0": 22, "iq3_0": 14, "fp4": 17}
SWIGLU_LIMIT = 10.0  # the official layer's clamp


def listed():
    return [
        # the smallest projection of the GEMV sweep: one vector, launch latency counts
        {"name": "gemv_q4_1024x4096_v1", "kind": "gemv", "fmt": "q4_0", "rows": 1024, "cols": 4096, "vectors": 1},
        # a short batch over a ragged projection (rows no multiple of a tile, 45 column pairs)
        {"name": "gemv_q5_5003x2880_v3", "kind": "gemv", "fmt": "q5_0", "rows": 5003, "cols": 2880, "vectors": 3},
        # the large projection of the GEMV sweep at its batch of 8
        {"name": "gemv_iq3_14336x4096_v8", "kind": "gemv", "fmt": "iq3_0", "rows": 14336, "cols": 4096, "vectors": 8},
        # a prompt's vectors through one square projection
        {"name": "gemv_q4_4096x4096_v64", "kind": "gemv", "fmt": "q4_0", "rows": 4096, "cols": 4096, "vectors": 64},
        # decode of one token: layers of the Qwen3-A3B shape replayed from a graph
        {"name": "stack_q4_12layers_t1", "kind": "stack", "fmt": "q4_0", "hidden": 2048, "inter": 768, "experts": 128,
         "k": 8, "tokens": 1, "layers": 12},
        # decode of 16 sequences through one such layer
        {"name": "layer_q4_t16", "kind": "layer", "fmt": "q4_0", "hidden": 2048, "inter": 768, "experts": 128, "k": 8,
         "tokens": 16, "shared": False},
        # a short prompt (odd length), 5-bit experts
        {"name": "layer_q5_t97", "kind": "layer", "fmt": "q5_0", "hidden": 2048, "inter": 768, "experts": 128, "k": 8,
         "tokens": 97, "shared": False},
        # prefill of a prompt chunk
        {"name": "layer_q4_t512", "kind": "layer", "fmt": "q4_0", "hidden": 2048, "inter": 768, "experts": 128, "k": 8,
         "tokens": 512, "shared": False},
        # decode of one token through the large split-FP4 layer with its shared expert
        {"name": "layer_fp4_shared_t1", "kind": "layer", "fmt": "fp4", "hidden": 7168, "inter": 2048, "experts": 256,
         "k": 8, "tokens": 1, "shared": True},
        # decode of 32 sequences in the official arithmetic (FP8 activations, FP8 shared expert)
        {"name": "official_fp4_t32", "kind": "official", "hidden": 7168, "inter": 2048, "experts": 256, "k": 8,
         "tokens": 32},
        # the host-in, host-out executor with its experts resident in the cache
        {"name": "executor_q4_resident", "kind": "executor", "fmt": "q4_0", "hidden": 2048, "inter": 768,
         "experts": 32, "k": 8},
        # packing a projection's weights
        {"name": "quantize_q4_4096x14336", "kind": "quantize", "fmt": "q4_0", "rows": 4096, "cols": 14336},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    u = rng.random()
    while True:
        if u < 0.35:
            fmt = rng.choice(list(FORMATS))
            step = 128 if fmt == "fp4" else 64
            c = {"kind": "gemv", "fmt": fmt, "rows": _log_int(rng, 300, 16384),
                 "cols": step * _log_int(rng, 512 // step, 14336 // step), "vectors": _log_int(rng, 1, 128)}
            if c["rows"] * c["cols"] * c["vectors"] <= 4096 * 14336 * 64 and _lanes(c["cols"]):
                return c
        elif u < 0.75:
            fmt = rng.choice(list(FORMATS))
            step = 128 if fmt == "fp4" else 64
            hidden = step * _log_int(rng, 512 // step, (7168 if fmt == "fp4" else 4096) // step)
            inter = step * _log_int(rng, 256 // step, 2048 // step)
            experts = _log_int(rng, 8, 256)
            c = {"kind": "layer", "fmt": fmt, "hidden": hidden, "inter": inter, "experts": experts,
                 "k": rng.randint(1, min(10, experts)), "tokens": _log_int(rng, 1, 512), "shared": rng.random() < 0.3}
            if _lanes(hidden) and _lanes(inter) and _routed_bytes(c) <= 9e9 and experts * _expert_bytes(c) <= 6e9:
                return c
        elif u < 0.85:
            experts = _log_int(rng, 8, 256)
            c = {"kind": "official", "hidden": rng.choice([1024, 1536, 2048, 2560, 3072, 4096, 5120, 7168]),
                 "inter": rng.choice([512, 768, 1024, 1408, 2048]), "experts": experts,
                 "k": rng.randint(1, min(8, experts)), "tokens": _log_int(rng, 1, 32)}
            return c
        elif u < 0.92:
            c = {"kind": "stack", "fmt": rng.choice(["q4_0", "q5_0", "iq3_0"]), "hidden": rng.choice([1024, 2048, 3072]),
                 "inter": 64 * rng.randint(4, 20), "experts": _log_int(rng, 8, 128), "k": rng.randint(1, 8),
                 "tokens": rng.randint(1, 4), "layers": rng.randint(2, 12)}
            if _lanes(c["inter"]):
                return c
        else:
            fmt = rng.choice(list(FORMATS))
            return {"kind": "quantize", "fmt": fmt, "rows": _log_int(rng, 300, 4096),
                    "cols": 32 * _log_int(rng, 16, 448)}


def _lanes(cols):
    """Column counts whose 64-wide pairs divide over 16 to 64 lanes, at most four each."""
    pairs = cols // 64
    return pairs <= 64 or any(pairs % d == 0 and pairs // d <= 4 for d in range(16, 65))


def _expert_bytes(c):
    fmt = c.get("fmt", "fp4")
    return 3 * c["hidden"] * c["inter"] // 32 * BLOCK_BYTES[fmt]


def _routed_bytes(c):
    return c["tokens"] * c["k"] * _expert_bytes(c)


# ------------------------------------------------------------------- backend
@functools.lru_cache(maxsize=None)
def _backend():
    be = HipBackend(0, 1)
    return be, MoeExecutor(be), QuantBackend(be)


# -------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + 17)


_SIGMA = 0.02
# block scales that cover +-2.2 sigma of weights ~ N(0, 0.02) over each format's codes
_BASE_SCALE = {"q4_0": 0.0062, "q5_0": 0.0029, "iq3_0": 0.0115}
_ZERO = {"q4_0": 8, "q5_0": 16, "iq3_0": 4}
_TOP = {"q4_0": 15, "q5_0": 31, "iq3_0": 7}
_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]
_FP4_UNIT = 2.0 ** -7


@functools.lru_cache(maxsize=None)
def _code_lut(fmt):
    """65536 quantiles of the weights' normal distribution as codes."""
    p = (torch.arange(65536, dtype=torch.float64) + 0.5) / 65536
    z = torch.erfinv(2 * p - 1) * math.sqrt(2.0) * _SIGMA
    if fmt == "fp4":
        levels = torch.tensor(_E2M1, dtype=torch.float64)
        code = (z.abs()[:, None] / _FP4_UNIT - levels).abs().argmin(1)
        code = code + 8 * (z < 0).long()
    else:
        code = (torch.round(z / _BASE_SCALE[fmt]) + _ZERO[fmt]).clamp(0, _TOP[fmt])
    return code.to(torch.uint8).cuda()


def _codes(fmt, gen, blocks):
    r = torch.empty((blocks, 32), dtype=torch.int32, device="cuda").random_(generator=gen)
    return _code_lut(fmt)[r & 0xFFFF]


def _nibbles(q):
    return q[:, 0::2] | (q[:, 1::2] << 4)


def _fill_blocks(fmt, gen, out):
    """out [blocks][block bytes] of one block format."""
    step = 1 << 21
    for b0 in range(0, out.shape[0], step):
        o = out[b0:b0 + step]
        n = o.shape[0]
        q = _codes(fmt, gen, n)
        s = (_BASE_SCALE[fmt] * torch.exp(0.15 * torch.randn(n, device="cuda", generator=gen))).to(torch.float16)
        o[:, 0:2] = s.view(torch.uint8).view(n, 2)
        if fmt == "q4_0":
            o[:, 2:18] = _nibbles(q)
        elif fmt == "q5_0":
            o[:, 6:22] = _nibbles(q & 15)
            bits = (q >> 4).view(n, 4, 8)
            o[:, 2:6] = (bits << torch.arange(8, dtype=torch.uint8, device="cuda")).sum(2).to(torch.uint8)
        else:
            low = (q & 3).view(n, 8, 4)
            o[:, 2:10] = (low << (2 * torch.arange(4, dtype=torch.uint8, device="cuda"))).sum(2).to(torch.uint8)
            high = (q >> 2).view(n, 4, 8)
            o[:, 10:14] = (high << torch.arange(8, dtype=torch.uint8, device="cuda")).sum(2).to(torch.uint8)


def _matrices(fmt, gen, n, rows, cols):
    """n matrices [rows][cols]: (weights [n][bytes], scales [n][bytes] or None)."""
    if fmt == "fp8":
        w = torch.empty((n, rows * cols), dtype=torch.uint8, device="cuda")
        for i in range(n):
            v = torch.randn(rows * cols, device="cuda", generator=gen).mul_(40.0).clamp_(-440.0, 440.0)
            w[i] = v.to(torch.float8_e4m3fn).view(torch.uint8)
        tiles = -(-rows // 128) * (cols // 128)
        s = torch.randint(115, 118, (n, tiles), device="cuda", generator=gen).to(torch.uint8)
        return w, s
    if fmt == "fp4":
        w = torch.empty((n, rows * cols // 2), dtype=torch.uint8, device="cuda")
        flat, step = w.view(-1, 16), 1 << 21
        for b0 in range(0, flat.shape[0], step):
            o = flat[b0:b0 + step]
            o[:] = _nibbles(_codes("fp4", gen, o.shape[0]))
        s = torch.randint(119, 122, (n, rows * cols // 32), dtype=torch.int32, device="cuda", generator=gen)
        return w, s.to(torch.uint8)
    w = torch.empty((n, rows * cols // 32 * BLOCK_BYTES[fmt]), dtype=torch.uint8, device="cuda")
    _fill_blocks(fmt, gen, w.view(-1, BLOCK_BYTES[fmt]))
    return w, None


def _expert_tensors(fmt, gen, n, hidden, inter):
    """(gate, up, down) of n experts, each (weights, scales)."""
    return (_matrices(fmt, gen, n, inter, hidden), _matrices(fmt, gen, n, inter, hidden),
            _matrices(fmt, gen, n, hidden, inter))


def _table(be, tensors):
    n = tensors[0][0].shape[0]

    def at(t, e):
        return 0 if t is None else t[e].data_ptr()
    return ExpertTable(be, [tuple(at(w, e) for w, _ in tensors) + tuple(at(s, e) for _, s in tensors)
                            for e in range(n)])


def _router(gen, experts, hidden):
    """Router weights and the bias of a Zipf(1.1) expert popularity."""
    w = torch.randn((experts, hidden), device="cuda", generator=gen) * 0.02
    rank = torch.argsort(torch.rand(experts, device="cuda", generator=gen)) + 1
    return w, (-1.1 * torch.log(rank.double())).float()


def _inputs(c, seed):
    """The tensors of a case (shared by prepare and exact)."""
    g, kind = _generator(seed), c["kind"]
    if kind == "gemv":
        w, s = _matrices(c["fmt"], g, 1, c["rows"], c["cols"])
        return {"w": w[0], "s": None if s is None else s[0],
                "x": torch.randn((c["vectors"], c["cols"]), device="cuda", generator=g)}
    if kind == "quantize":
        return {"m": torch.randn((c["rows"], c["cols"]), device="cuda", generator=g) * _SIGMA}
    hidden, inter, experts = c["hidden"], c["inter"], c["experts"]
    if kind in ("layer", "stack"):
        layers = [_expert_tensors(c["fmt"], g, experts, hidden, inter) for _ in range(c.get("layers", 1))]
        routers = [_router(g, experts, hidden) for _ in layers]
        shared = _expert_tensors(c["fmt"], g, 1, hidden, inter) if c.get("shared") else None
        return {"layers": layers, "routers": routers, "shared": shared,
                "x": torch.randn((c["tokens"], hidden), device="cuda", generator=g)}
    tokens = c.get("tokens", 1)
    d = {"experts": _expert_tensors(c.get("fmt", "fp4"), g, experts, hidden, inter),
         "shared": _expert_tensors("fp8", g, 1, hidden, inter) if kind == "official" else None,
         "x": torch.randn((tokens, hidden), device="cuda", generator=g)}
    _, bias = _router(g, experts, 1)
    logits = torch.randn((tokens, experts), device="cuda", generator=g) + bias
    top, ids = torch.topk(torch.softmax(logits, 1), c["k"], dim=1)
    d["ids"], d["weights"] = ids.to(torch.int32).contiguous(), (top / top.sum(1, keepdim=True)).contiguous()
    return d


class _Graph:
    def __init__(self, be, enqueue):
        self.be, self.g = be, C.c_void_p()
        check(be.L.objeta_hip_graph_begin_capture(be.ctx, None))
        enqueue()
        check(be.L.objeta_hip_graph_end_capture(be.ctx, None, C.byref(self.g)))

    def launch(self):
        check(self.be.L.objeta_hip_graph_launch(self.be.ctx, self.g, None))

    def __del__(self):
        if self.g and self.be.ctx:
            self.be.synchronize()
            self.be.L.objeta_hip_graph_destroy(self.be.ctx, self.g)


def prepare(case, seed):
    be, moe, quant = _backend()
    c, d, kind = case, _inputs(case, seed), case["kind"]
    state = {"case": c, "in": d}

    def empty(*shape, dtype=torch.float32):
        return torch.empty(shape, dtype=dtype, device="cuda")
    if kind == "gemv":
        state["y"] = empty(c["vectors"], c["rows"])
        state["shape"] = QGemvShape.new(FORMATS[c["fmt"]], c["rows"], c["cols"])
    elif kind == "quantize":
        state["out"] = empty(c["rows"] * c["cols"] // 32 * BLOCK_BYTES[c["fmt"]], dtype=torch.uint8)
    elif kind in ("layer", "stack"):
        n, t, k = len(d["layers"]), c["tokens"], c["k"]
        state["tables"] = [_table(be, lay) for lay in d["layers"]]
        state["shared"] = None if d["shared"] is None else _table(be, d["shared"])
        state["out"] = empty(t, c["hidden"])
        state["ids"], state["weights"] = empty(n, t, k, dtype=torch.int32), empty(n, t, k)
        if kind == "stack":
            torch.cuda.synchronize()
            _layers(state)  # workspaces are made outside the capture
            be.synchronize()
            state["graph"] = _Graph(be, lambda: _layers(state))
    elif kind == "official":
        state["table"], state["shared"] = _table(be, d["experts"]), _table(be, d["shared"])
        state["out"] = empty(c["tokens"], c["hidden"])
    else:
        host = [w.cpu().numpy() for w, _ in d["experts"]]
        state["host"] = HostExpertSet([tuple(m[e] for m in host) for e in range(c["experts"])])
        state["cache"] = ExpertCache(c["experts"] * _expert_bytes(c), be)
        state["x"] = d["x"][0].cpu().numpy()
        state["selected"] = [(int(i), float(w)) for i, w in zip(d["ids"][0].cpu(), d["weights"][0].cpu())]
    torch.cuda.synchronize()
    return state


def _layers(s):
    moe, c, d = _backend()[1], s["case"], s["in"]
    out = s["out"].data_ptr()
    for i, (table, (w, b)) in enumerate(zip(s["tables"], d["routers"])):
        # a stack updates its residual stream in place from the second layer on; a layer of
        # its own returns the experts' sum, which the program's next operation adds
        x = d["x"].data_ptr() if i == 0 else out
        moe.layer_device(FORMATS[c["fmt"]], table, w.data_ptr(), b.data_ptr(), c["k"], c["tokens"], x,
                         x if c["kind"] == "stack" else None, out,
                         s["ids"][i].data_ptr(), s["weights"][i].data_ptr(), c["hidden"], c["inter"], c["hidden"],
                         shared=s["shared"])


def run(state):
    be, moe, quant = _backend()
    c, d, kind = state["case"], state["in"], state["case"]["kind"]
    if kind == "gemv":
        if c["fmt"] == "fp4":
            quant.launch_kernel_split_fp4(None, d["w"].data_ptr(), d["s"].data_ptr(), d["x"].data_ptr(),
                                          state["y"].data_ptr(), c["rows"], c["cols"], c["vectors"])
        else:
            quant.launch_kernel(FORMATS[c["fmt"]], None, d["w"].data_ptr(), d["x"].data_ptr(), state["y"].data_ptr(),
                                state["shape"], c["vectors"])
        return state["y"]
    if kind == "quantize":
        check(be.L.objeta_hip_quantize_matrix_device(be.ctx, int(FORMATS[c["fmt"]]), None,
                                                     C.c_void_p(d["m"].data_ptr()), c["rows"], c["cols"],
                                                     C.c_void_p(state["out"].data_ptr())))
        return state["out"]
    if kind == "layer":
        _layers(state)
        return state["out"], state["ids"], state["weights"]
    if kind == "stack":
        state["graph"].launch()
        return state["out"], state["ids"], state["weights"]
    if kind == "official":
        moe.official_fp4_device(state["table"], d["ids"].data_ptr(), d["weights"].data_ptr(), c["tokens"], c["k"],
                                d["x"].data_ptr(), state["out"].data_ptr(), c["hidden"], c["inter"], c["hidden"],
                                swiglu_limit=SWIGLU_LIMIT, shared_fp8=state["shared"])
        return state["out"]
    out, _ = moe.execute_selected_moe_cuda(quant, None, state["host"], state["selected"], state["x"], c["hidden"],
                                           c["inter"], c["hidden"], 0, state["cache"], FORMATS[c["fmt"]])
    return out


# ------------------------------------------------------------------- 64 bits
def _f8_values():
    """E4M3 codes as the format defines them here: field 0 is mant * 2^-5, 15 is +-448."""
    v = []
    for code in range(256):
        e, m = (code >> 3) & 15, code & 7
        a = m / 32.0 if e == 0 else 448.0 if e == 15 else (1 + m / 8.0) * 2.0 ** (e - 7)
        v.append(-a if code & 128 else a)
    return torch.tensor(v, dtype=torch.float64, device="cuda")


def _matrix64(fmt, w, s, rows, cols):
    """The float64 values [rows][cols] of a packed matrix."""
    if fmt == "fp8":
        v = _f8_values()[w.int()].view(rows, cols)
        t = torch.exp2(s.double() - 127).view(-1, cols // 128)
        return v * t.repeat_interleave(128, 0)[:rows].repeat_interleave(128, 1)
    if fmt == "fp4":
        levels = torch.tensor(_E2M1 + [-v for v in _E2M1], dtype=torch.float64, device="cuda")
        v = torch.stack((levels[(w & 15).int()], levels[(w >> 4).int()]), 1)
        return (v.view(-1, 32) * torch.exp2(s.double() - 127)[:, None]).view(rows, cols)
    b = w.view(-1, BLOCK_BYTES[fmt])
    scale = b[:, 0:2].contiguous().view(torch.float16).double()
    nib = b[:, 2:18] if fmt == "q4_0" else b[:, 6:22]
    eight = torch.arange(8, dtype=torch.uint8, device="cuda")
    if fmt == "iq3_0":
        q = ((b[:, 2:10, None] >> (2 * torch.arange(4, dtype=torch.uint8, device="cuda"))) & 3).reshape(-1, 32)
        q = q + (((b[:, 10:14, None] >> eight) & 1) << 2).reshape(-1, 32)
    else:
        q = torch.stack((nib & 15, nib >> 4), 2).reshape(-1, 32)
        if fmt == "q5_0":
            q = q + (((b[:, 2:6, None] >> eight) & 1) << 4).reshape(-1, 32)
    return ((q.double() - _ZERO[fmt]) * scale).view(rows, cols)


def _expert64(fmt, tensors, e, hidden, inter):
    dims = ((inter, hidden), (inter, hidden), (hidden, inter))
    return [_matrix64(fmt, w[e], None if s is None else s[e], r, c) for (w, s), (r, c) in zip(tensors, dims)]


def _fp8_round(x):
    """Activations (float32 [rows][cols]) through FP8 codes with one scale per 128: the
    dequantized values, in float64."""
    v = x.view(x.shape[0], -1, 128)
    amax = v.abs().amax(2, keepdim=True).clamp(min=1e-4)
    scale = torch.exp2(torch.ceil(torch.log2((amax * (1.0 / 448.0)).double()).float().double()))
    a = (v.double() / scale).float().clamp(-448.0, 448.0)
    m, e = torch.frexp(a.abs())
    mant = torch.floor((2 * m.double() - 1) * 8 + 0.5)
    ex = e.double() - 1
    ex = ex + (mant >= 8)
    mant = torch.where(mant >= 8, torch.zeros_like(mant), mant)
    big = torch.where(ex > 7, torch.full_like(mant, 240.0), (1 + mant / 8) * torch.exp2(ex))
    q = torch.where(ex == -7, mant / 32, big)  # exponent field 0
    q = torch.where(a.abs() < 1.0 / 128, torch.zeros_like(q), q)
    q = torch.where(a.abs() >= 448, torch.full_like(q, 448.0), q)
    return (torch.copysign(q, a.double()) * scale).view(x.shape)


def _experts64(fmt, tensors, ids, weights, x, hidden, inter, official):
    """sum_j w_j down_j(act_j) over each token's selection."""
    y = torch.zeros_like(x)
    for e in torch.unique(ids).tolist():
        t, j = torch.nonzero(ids == e, as_tuple=True)
        y.index_add_(0, t, weights[t, j].double()[:, None] *
                     _mlp64(_expert64(fmt, tensors, e, hidden, inter), x[t], official))
    return y


def _mlp64(mats, x, official):
    g, u = x @ mats[0].T, x @ mats[1].T
    if official:
        u = u.clamp(-SWIGLU_LIMIT, SWIGLU_LIMIT)
    a = g * torch.sigmoid(g) * u
    return (_fp8_round(a.float()) if official else a) @ mats[2].T


def exact(case, seed):
    c, d, kind = case, _inputs(case, seed), case["kind"]
    if kind == "quantize":
        return None
    if kind == "gemv":
        return d["x"].double() @ _matrix64(c["fmt"], d["w"], d["s"], c["rows"], c["cols"]).T
    hidden, inter = c["hidden"], c["inter"]
    if kind in ("official", "executor"):
        official = kind == "official"
        x = _fp8_round(d["x"]) if official else d["x"].double()
        y = _experts64(c.get("fmt", "fp4"), d["experts"], d["ids"], d["weights"], x, hidden, inter, official)
        if official:
            return y + _mlp64(_expert64("fp8", d["shared"], 0, hidden, inter), x, True)
        return y[0].cpu().numpy()
    h, ids_all, w_all = d["x"].double(), [], []
    for lay, (w, b) in zip(d["layers"], d["routers"]):
        p = torch.softmax(h @ w.double().T + b.double(), 1)
        top, ids = torch.topk(p, c["k"], dim=1)
        top = top / top.sum(1, keepdim=True)
        y = _experts64(c["fmt"], lay, ids, top, h, hidden, inter, False)
        if d["shared"] is not None:
            y = y + _mlp64(_expert64(c["fmt"], d["shared"], 0, hidden, inter), h, False)
        h = h + y if kind == "stack" else y
        ids_all.append(ids.to(torch.int32))
        w_all.append(top)
    return h, torch.stack(ids_all), torch.stack(w_all)


# ------------------------------------------------------------ work, tolerance
def _distinct(c):
    """Experts that a call selects, from the distribution that the inputs follow."""
    r = np.random.default_rng(11)
    spread = 0.02 * math.sqrt(c["hidden"]) if c["kind"] in ("layer", "stack") else 1.0
    n = c["experts"]
    logits = spread * r.standard_normal((c.get("tokens", 1), n)) - 1.1 * np.log(np.arange(1, n + 1))
    return len(np.unique(np.argsort(-logits, axis=1)[:, :c["k"]]))


def work(case):
    c, kind = case, case["kind"]
    if kind == "gemv":
        n = c["rows"] * c["cols"]
        return {"bytes": n // 32 * BLOCK_BYTES[c["fmt"]] + 4 * c["vectors"] * (c["rows"] + c["cols"]),
                "flops": 2 * n * c["vectors"]}
    if kind == "quantize":
        n = c["rows"] * c["cols"]
        return {"bytes": 4 * n + n // 32 * BLOCK_BYTES[c["fmt"]], "flops": 4 * n}
    hidden, inter, t, k = c["hidden"], c["inter"], c.get("tokens", 1), c["k"]
    b = _distinct(c) * _expert_bytes(c) + 8 * t * hidden
    f = 6 * t * k * hidden * inter
    if kind in ("layer", "stack"):
        b += 4 * c["experts"] * hidden + 8 * t * k
        f += 2 * t * c["experts"] * hidden
        if c.get("shared"):
            b += _expert_bytes(c)
            f += 6 * t * hidden * inter
    elif kind == "official":
        b += 3 * hidden * inter
        f += 6 * t * hidden * inter
    n = c.get("layers", 1)
    return {"bytes": n * b, "flops": n * f}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    # 32-bit sums over some thousand products differ by about 1e-7 from the exact ones
    # (2-norm), a stack's by a few times that; the official layer's intermediates pass
    # through FP8 codes, where another order of a sum moves a code now and then (2e-6 and
    # more); a selection may differ where two experts' logits agree to 32 bits
    if kind == "official":
        return {"rel": 1e-4, "max": 5e-3}
    if kind == "stack":
        return {"rel": 4e-6, "max": 1e-4, "differ": 0.002}
    if kind == "layer":
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.002}
    return {"rel": 1e-6, "max": 1e-5}
