"""What a user of this package has it do on the GPU, as cases to time and to compare.

Every case goes through the public entry points of dynet_amd, fp32 throughout (the package's one data type): the
language-model training step of the baseline on the fused path and, at another size, node by node; scoring a batch of
sentences; generating a token; a single LSTM cell, forward and backward, through its nodes; the elementwise sweep;
LayerNorm; the embedding lookup with its sparse update; PickNegLogSoftmax; attention over a batch; and a feed-forward
classifier's training step.  One Device serves the whole process, as in a user's program; parameters, gradients and
inputs of the node-level cases live in torch tensors whose addresses the calls are given.

Gradients are zeroed at the start of a backward pass, as the executor does, and scratch goes back to its pool at the
end of a pass, as a node's scratch does.
"""
import math
import weakref

import numpy as np
import torch

from dynet_amd import Device, DevTensor, lib
from dynet_amd.lm import LstmLM
from dynet_amd.synth import zipf_ids

# ---------------------------------------------------------------------------------------------------------------
# the device and what a state holds of its pools
# ---------------------------------------------------------------------------------------------------------------
_POOL_MB = (6144, 6144, 4096, 8192)
_device = None
_taken = []  # one entry a live state, oldest first: [pool levels before it, still alive]


def device():
    global _device
    if _device is None:
        _device = Device(0, mem_mb=_POOL_MB)
    return _device


def _levels():
    return [device().pool(w).used() for w in range(4)]


def _give_back(entry):
    entry[1] = False
    while _taken and not _taken[-1][1]:
        for w, level in enumerate(_taken.pop()[0]):
            device().pool(w).set_used(level)


class State:
    """Everything one prepared case keeps.  What it allocated from the pools goes back when it is dropped."""

    def __init__(self, case):
        entry = [_levels(), True]
        _taken.append(entry)
        self._finalizer = weakref.finalize(self, _give_back, entry)
        self._finalizer.atexit = False
        self.case = case
        self.dev = device()
        self.scs = self.dev.pool(lib.POOL_SCS)
        self._keep = []

    def t(self, tensor):
        """A torch tensor as the package's tensor (same memory)."""
        self._keep.append(tensor)
        dtype = {torch.int32: np.uint32, torch.int64: np.int64}.get(tensor.dtype, np.float32)
        return DevTensor(self.dev, tensor.data_ptr(), tensor.shape, dtype)

    def new(self, *shape, dtype=torch.float32):
        """An output buffer: (torch tensor, the package's tensor)."""
        x = torch.zeros(shape, dtype=dtype, device="cuda")
        return x, self.t(x)

    def scratch_level(self):
        self.scs_level = self.scs.used()

    def scratch_back(self):
        self.scs.set_used(self.scs_level)


class _Memory:
    """Pool memory for torch: the device's, for as long as the process runs."""

    def __init__(self, t):
        self.__cuda_array_interface__ = {"shape": t.shape, "typestr": "<f4", "data": (t.ptr, False), "version": 2}


def _view(t):
    return torch.as_tensor(_Memory(t), device="cuda")


def _generators(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g, np.random.default_rng(seed)


def _normal(g, *shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std


def _uniform(g, lo, hi, *shape):
    return torch.rand(shape, generator=g, device="cuda", dtype=torch.float32) * (hi - lo) + lo


def _glorot(g, rows, cols):
    """A rows x cols matrix, column-major (torch shape reversed)."""
    s = math.sqrt(6.0 / (rows + cols))
    return _uniform(g, -s, s, cols, rows)


class Slab:
    """Tensors one behind the other in one buffer, each on a 256-byte boundary: gradients that one call zeroes."""

    def __init__(self, s, shapes):
        pad = [(int(np.prod(sh)) + 63) // 64 * 64 for sh in shapes.values()]
        self.torch = torch.zeros(sum(pad), device="cuda")
        self.all = s.t(self.torch)
        self.views, self.dev, at = {}, {}, 0
        for (name, sh), n in zip(shapes.items(), pad):
            self.views[name] = self.torch[at:at + int(np.prod(sh))].view(*sh)
            self.dev[name] = s.t(self.views[name])
            at += n


# ---------------------------------------------------------------------------------------------------------------
# the language model: training step (fused path; node by node), scoring
# ---------------------------------------------------------------------------------------------------------------
def _lm(case, seed, **how):
    s = State(case)
    V, E, H, L, B, T = (case[k] for k in ("V", "E", "H", "L", "B", "T"))
    s.lm = LstmLM(s.dev, V, E, H, L, B, T, seed=seed, lr=0.1, clip=5.0, **how)
    rng = np.random.default_rng(seed)
    s.tokens = zipf_ids(rng, (T + 1) * B, V).reshape(T + 1, B)
    return s


def _lm_flops(case, passes):
    V, E, H, L, B, T = (case[k] for k in ("V", "E", "H", "L", "B", "T"))
    macs = T * B * (sum(4 * H * ((E if l == 0 else H) + H) for l in range(L)) + H * V)
    return 2.0 * passes * macs


def _lm_weights(case):
    V, E, H, L = (case[k] for k in ("V", "E", "H", "L"))
    return sum(4 * H * ((E if l == 0 else H) + H + 1) for l in range(L)) + V * H + V


def prepare_train(case, seed):
    nodes = case["path"] == "nodes"
    s = _lm(case, seed, path=case["path"], dropout=case["dropout"], time_batched=not nodes, defer_weight_grads=nodes)
    s.dev.reset_rng(seed & 0x7FFFFFFF or 1)
    weakref.finalize(s, s.lm.capture().destroy).atexit = False
    s.out = [_view(t) for t in [s.lm.loss, s.lm.logits] + [s.lm.p[n] for n in sorted(s.lm.p)]]
    return s


def run_train(s):
    s.lm.step(s.tokens, read_loss=False)
    return s.out


def work_train(case):
    V, E, H, L, B, T = (case[k] for k in ("V", "E", "H", "L", "B", "T"))
    # weights read and written once, so the embedding rows; the logits written (their gradient need not be)
    rows = min(V, T * B)
    return {"bytes": 4.0 * (2 * _lm_weights(case) + 2 * rows * E + T * B * V) + 8.0 * T * B, "flops": _lm_flops(case, 3)}


def prepare_score(case, seed):
    s = _lm(case, seed)
    s.scratch_level()
    s.out = [_view(t) for t in (s.lm.loss, s.lm.errs, s.lm.logits)]
    return s


def run_score(s):
    s.lm.stage(s.tokens)
    s.lm.forward()
    s.scratch_back()
    return s.out


def work_score(case):
    V, E, T, B = (case[k] for k in ("V", "E", "T", "B"))
    return {"bytes": 4.0 * (_lm_weights(case) + min(V, T * B) * E + T * B * V + T * B) + 8.0 * T * B,
            "flops": _lm_flops(case, 1)}


# ---------------------------------------------------------------------------------------------------------------
# generating: one token for each of B sentences.  The program reads the tokens (it prints them and looks for the end
# of a sentence) and feeds them back.
# ---------------------------------------------------------------------------------------------------------------
def prepare_decode(case, seed):
    s = State(case)
    d = s.dev
    V, E, H, L, B = (case[k] for k in ("V", "E", "H", "L", "B"))
    g, rng = _generators(seed)
    s.table = s.t(_uniform(g, -math.sqrt(3.0 / E), math.sqrt(3.0 / E), V, E))
    s.R, s.bias = s.t(_glorot(g, V, H)), s.t(_uniform(g, -0.1, 0.1, V))
    s.tokens = zipf_ids(rng, B, V)
    s.ids, s.best = s.new(B, dtype=torch.int32)[1], s.new(B, dtype=torch.int64)[1]
    s.emb = s.new(B, E)[1]
    s.logits_t, s.logits = s.new(B, V)
    s.layers, s.state_t = [], []
    s.packed = E % 128 == 0 and H % 128 == 0 and d.lstm_step_supported(H, B)
    for l in range(L):
        d_in = E if l == 0 else H
        Wx, Wh, b = s.t(_glorot(g, 4 * H, d_in)), s.t(_glorot(g, 4 * H, H)), s.t(_normal(g, 4 * H, std=0.1))
        if s.packed:  # weights laid out once for the one-launch cell
            pWx, pWh = s.new(4 * H * d_in)[1], s.new(4 * H * H)[1]
            d.lstm_pack_input(d_in, H, Wx, pWx)
            d.lstm_pack_recurrent(H, Wh, pWh)
            Wx, Wh = pWx, pWh
        pairs = []  # the state before and after a token, used in turn
        for k in range(2):
            h_t, c_t = _normal(g, B, H, std=0.3), _normal(g, B, H, std=0.5)
            s.state_t.append((h_t, c_t))
            pairs.append((s.t(h_t), s.t(c_t)))
        s.layers.append((d_in, Wx, Wh, b, s.new(B, 4 * H)[1], pairs))
    s.at = 0
    s.scratch_level()
    d.sync()
    torch.cuda.synchronize()
    return s


def run_decode(s):
    d, case = s.dev, s.case
    V, E, H, B = case["V"], case["E"], case["H"], case["B"]
    d.lookup_forward(s.tokens, s.ids, E, V, s.table, s.emb)
    x, old, new = s.emb, s.at, s.at ^ 1
    for d_in, Wx, Wh, b, gates, pairs in s.layers:
        (h0, c0), (h1, c1) = pairs[old], pairs[new]
        if s.packed:
            d.lstm_step_forward_x(d_in, H, B, Wx, x, Wh, h0, b, c0, gates, c1, h1)
        else:
            d.lstm_gates_forward([x], [d_in], H, B, h0, Wx, Wh, b, gates)
            d.lstm_c_forward(H, B, c0, gates, c1)
            d.lstm_h_forward(H, B, c1, gates, h1)
        x = h1
    d.affine_forward(V, B, H, s.bias, s.R, x, s.logits)
    d.argmax_cols(V, B, s.logits, s.best)
    s.tokens = s.best.numpy().astype(np.uint32)
    s.scratch_back()
    s.at = new
    return [s.logits_t, s.tokens] + [t for k, pair in enumerate(s.state_t) if k % 2 == new for t in pair]


def work_decode(case):
    V, E, H, L, B = (case[k] for k in ("V", "E", "H", "L", "B"))
    w = _lm_weights(case)
    return {"bytes": 4.0 * (w + B * (E + 4 * L * H + V + 2)), "flops": 2.0 * B * w}


# ---------------------------------------------------------------------------------------------------------------
# one LSTM cell through its three nodes, forward and every backward argument
# ---------------------------------------------------------------------------------------------------------------
def prepare_cell(case, seed):
    s = State(case)
    I, H, B = case["I"], case["H"], case["B"]
    g, _ = _generators(seed)
    s.x, s.h, s.c = (s.t(_normal(g, B, n)) for n in (I, H, H))
    s.Wx, s.Wh = s.t(_glorot(g, 4 * H, I)), s.t(_glorot(g, 4 * H, H))
    s.b = s.t(torch.zeros(4 * H, device="cuda"))
    s.dh = s.t(_normal(g, B, H))
    s.gates_t, s.gates = s.new(B, 4 * H)
    s.c2_t, s.c2 = s.new(B, H)
    s.h2_t, s.h2 = s.new(B, H)
    s.dpre = s.new(B, 4 * H)[1]
    s.grads = Slab(s, {"gates": (B, 4 * H), "c2": (B, H), "c": (B, H), "x": (B, I), "h": (B, H), "Wx": (I, 4 * H),
                       "Wh": (H, 4 * H), "b": (4 * H,)})
    s.scratch_level()
    torch.cuda.synchronize()
    return s


def run_cell(s):
    d = s.dev
    I, H, B = s.case["I"], s.case["H"], s.case["B"]
    d.lstm_gates_forward([s.x], [I], H, B, s.h, s.Wx, s.Wh, s.b, s.gates)
    d.lstm_c_forward(H, B, s.c, s.gates, s.c2)
    d.lstm_h_forward(H, B, s.c2, s.gates, s.h2)
    q = s.grads.dev
    d.zero(s.grads.all)
    d.lstm_h_backward(H, B, s.c2, s.gates, s.dh, 0, q["c2"])
    d.lstm_h_backward(H, B, s.c2, s.gates, s.dh, 1, q["gates"])
    d.lstm_c_backward(H, B, s.c, s.gates, q["c2"], 0, q["c"])
    d.lstm_c_backward(H, B, s.c, s.gates, q["c2"], 1, q["gates"])
    d.lstm_gates_dpre(H, B, s.gates, q["gates"], s.dpre)
    for i, name in enumerate(("x", "h", "Wx", "Wh", "b")):
        d.lstm_gates_backward([s.x], [I], H, B, s.h, s.Wx, s.Wh, s.gates, q["gates"], i, q[name], dpre=s.dpre)
    s.scratch_back()
    return [s.gates_t, s.c2_t, s.h2_t, s.grads.views]


def work_cell(case):
    I, H, B = case["I"], case["H"], case["B"]
    w = 4 * H * (I + H + 1)
    return {"bytes": 4.0 * (2 * w + B * (I + 3 * H + 4 * H + 2 * H + 4 * H + 3 * H + I)), "flops": 6.0 * B * 4 * H * (I + H)}


# ---------------------------------------------------------------------------------------------------------------
# elementwise nodes and sum_batches, forward and backward
# ---------------------------------------------------------------------------------------------------------------
_OPS = (lib.OP_TANH, lib.OP_LOGISTIC, lib.OP_RECTIFY)


def prepare_elementwise(case, seed):
    s = State(case)
    n, bd = case["n"], case["bd"]
    g, _ = _generators(seed)
    s.a, s.b, s.dy = (s.t(_normal(g, bd, n)) for _ in range(3))
    s.dsum = s.t(_normal(g, n))
    s.y = [s.new(bd, n) for _ in range(4)]
    s.sum_t, s.sum = s.new(n)
    s.grads = Slab(s, {k: (bd, n) for k in ("tanh", "logistic", "rectify", "a", "b", "sum")})
    s.scratch_level()
    torch.cuda.synchronize()
    return s


def run_elementwise(s):
    d, n, bd = s.dev, s.case["n"], s.case["bd"]
    for op, (_, y) in zip(_OPS, s.y):
        d.unary_forward(op, s.a, y)
    d.cmult_forward(n, bd, bd, s.a, s.b, s.y[3][1])
    d.sum_batches_forward(n, bd, s.a, s.sum)
    q = s.grads.dev
    d.zero(s.grads.all)
    for op, (_, y), name in zip(_OPS, s.y, ("tanh", "logistic", "rectify")):
        d.unary_backward(op, y, s.dy, q[name])
    d.cmult_backward(n, bd, bd, s.a, s.b, s.dy, 0, q["a"])
    d.cmult_backward(n, bd, bd, s.a, s.b, s.dy, 1, q["b"])
    d.sum_batches_backward(n, bd, s.dsum, q["sum"])
    s.scratch_back()
    return [[y for y, _ in s.y], s.sum_t, s.grads.views]


def work_elementwise(case):
    m = case["n"] * case["bd"]
    return {"bytes": 4.0 * (3 * m + 2 * case["n"] + 4 * m + 6 * m), "flops": 20.0 * m}


# ---------------------------------------------------------------------------------------------------------------
# LayerNorm, forward and backward
# ---------------------------------------------------------------------------------------------------------------
def prepare_layer_norm(case, seed):
    s = State(case)
    n, bd = case["n"], case["bd"]
    g, _ = _generators(seed)
    s.x, s.dy = s.t(_normal(g, bd, n)), s.t(_normal(g, bd, n))
    s.g, s.b = s.t(_uniform(g, 0.5, 1.5, n)), s.t(_normal(g, n, std=0.1))
    s.y_t, s.y = s.new(bd, n)
    s.grads = Slab(s, {"x": (bd, n), "g": (n,), "b": (n,)})
    s.scratch_level()
    torch.cuda.synchronize()
    return s


def run_layer_norm(s):
    d, n, bd = s.dev, s.case["n"], s.case["bd"]
    d.layer_norm_forward(n, bd, s.x, s.g, s.b, s.y)
    d.zero(s.grads.all)
    q = s.grads.dev
    d.layer_norm_backward(n, bd, s.x, s.g, s.dy, q["x"], q["g"], q["b"])
    s.scratch_back()
    return [s.y_t, s.grads.views]


def work_layer_norm(case):
    m = case["n"] * case["bd"]
    return {"bytes": 4.0 * (4 * m + 4 * case["n"]), "flops": 20.0 * m}


# ---------------------------------------------------------------------------------------------------------------
# embedding lookup: gather, scatter-add of its gradient, update of the touched rows
# ---------------------------------------------------------------------------------------------------------------
def prepare_lookup(case, seed):
    s = State(case)
    V, D, n = case["V"], case["D"], case["n"]
    g, rng = _generators(seed)
    s.table_t = _uniform(g, -0.1, 0.1, V, D)
    s.table, s.dtable = s.t(s.table_t), s.new(V, D)[1]
    s.ids_host = zipf_ids(rng, n, V)
    s.ids = s.new(n, dtype=torch.int32)[1]
    s.dy = s.t(_normal(g, n, D, std=0.01))
    s.fx_t, s.fx = s.new(n, D)
    s.scale = s.t(torch.ones(1, device="cuda"))
    s.plan, s.plan_ws, s.plan_bytes = s.dev.lookup_plan_buffers(n, V)
    s.scratch_level()
    torch.cuda.synchronize()
    return s


def run_lookup(s):
    d = s.dev
    V, D, n = s.case["V"], s.case["D"], s.case["n"]
    d.lookup_forward(s.ids_host, s.ids, D, V, s.table, s.fx)
    d.lookup_build_plan_into(s.ids, V, s.plan, s.plan_ws, s.plan_bytes)
    d.lookup_accumulate_grads_planned(n, s.plan, D, V, s.dy, s.dtable)
    d.sgd_update_rows(n, s.plan, D, V, s.table, s.dtable, 0.1, s.scale)
    s.scratch_back()
    return [s.fx_t, s.table_t]


def work_lookup(case):
    V, D, n = case["V"], case["D"], case["n"]
    p = np.arange(1, V + 1, dtype=np.float64) ** -1.1
    rows = float(np.sum(1.0 - np.exp(n * np.log1p(-p / p.sum()))))  # expected number of different ids
    return {"bytes": 4.0 * (2 * n * D + 2 * rows * D + n), "flops": float(n * D + 2 * rows * D)}


# ---------------------------------------------------------------------------------------------------------------
# PickNegLogSoftmax over a vocabulary, forward and backward
# ---------------------------------------------------------------------------------------------------------------
def prepare_pnls(case, seed):
    s = State(case)
    V, B = case["V"], case["B"]
    g, rng = _generators(seed)
    s.x = s.t(_normal(g, B, V, std=2.0))
    s.labels = rng.integers(0, V, B).astype(np.uint32)
    s.aux = s.new(3 * B)[1]
    s.fx_t, s.fx = s.new(B)
    s.dy = s.t(torch.ones(B, device="cuda"))
    s.dx_t, s.dx = s.new(B, V)
    s.scratch_level()
    torch.cuda.synchronize()
    return s


def run_pnls(s):
    d, V, B = s.dev, s.case["V"], s.case["B"]
    d.pnls_forward(V, B, s.x, s.labels, s.aux, s.fx)
    d.zero(s.dx)
    d.pnls_backward(V, B, s.x, s.aux, s.dy, s.dx)
    s.scratch_back()
    return [s.fx_t, s.dx_t]


def work_pnls(case):
    m = case["V"] * case["B"]
    return {"bytes": 4.0 * (2 * m + 3 * case["B"]), "flops": 6.0 * m}


# ---------------------------------------------------------------------------------------------------------------
# dot-product attention of one decoder state a sentence over its T encoder states, forward and backward
# ---------------------------------------------------------------------------------------------------------------
def prepare_attention(case, seed):
    s = State(case)
    H, T, B = case["H"], case["T"], case["B"]
    g, _ = _generators(seed)
    s.enc, s.q, s.dctx = s.t(_normal(g, B, T, H, std=0.5)), s.t(_normal(g, B, H, std=0.2)), s.t(_normal(g, B, H))
    s.e = s.new(B, T)[1]
    s.a_t, s.a = s.new(B, T)
    s.ctx_t, s.ctx = s.new(B, H)
    s.grads = Slab(s, {"enc": (B, T, H), "q": (B, H), "a": (B, T), "e": (B, T)})
    s.scratch_level()
    torch.cuda.synchronize()
    return s


def run_attention(s):
    d = s.dev
    H, T, B = s.case["H"], s.case["T"], s.case["B"]
    mm = d.gemm_strided_batched
    mm(1, 0, T, 1, H, s.enc, T * H, s.q, H, 0.0, s.e, T, B)        # e = enc^T q
    d.softmax_forward(T, B, s.e, s.a)
    mm(0, 0, H, 1, T, s.enc, T * H, s.a, T, 0.0, s.ctx, H, B)      # ctx = enc a
    g = s.grads.dev
    d.zero(s.grads.all)
    mm(1, 0, T, 1, H, s.enc, T * H, s.dctx, H, 1.0, g["a"], T, B)  # da += enc^T dctx
    mm(0, 1, H, T, 1, s.dctx, H, s.a, T, 1.0, g["enc"], T * H, B)  # denc += dctx a^T
    d.softmax_backward(T, B, s.a, g["a"], g["e"])
    mm(0, 0, H, 1, T, s.enc, T * H, g["e"], T, 1.0, g["q"], H, B)  # dq += enc de
    mm(0, 1, H, T, 1, s.q, H, g["e"], T, 1.0, g["enc"], T * H, B)  # denc += q de^T
    s.scratch_back()
    return [s.a_t, s.ctx_t, s.grads.views]


def work_attention(case):
    H, T, B = case["H"], case["T"], case["B"]
    return {"bytes": 4.0 * B * (2 * H * T + 4 * H + 5 * T), "flops": 12.0 * B * H * T}


# ---------------------------------------------------------------------------------------------------------------
# a feed-forward classifier: three affine layers, dropout, clipped SGD step
# ---------------------------------------------------------------------------------------------------------------
def prepare_classifier(case, seed):
    s = State(case)
    D, H, C, B = case["D"], case["H"], case["C"], case["B"]
    g, rng = _generators(seed)
    shapes = {"W1": (D, H), "b1": (H,), "W2": (H, H), "b2": (H,), "W3": (H, C), "b3": (C,)}
    s.p, s.g = Slab(s, shapes), Slab(s, shapes)
    for name in ("W1", "W2", "W3"):
        cols, rows = shapes[name]
        s.p.views[name].copy_(_glorot(g, rows, cols))
    s.x = s.t(_uniform(g, 0.0, 1.0, B, D))
    s.labels = rng.integers(0, C, B).astype(np.uint32)
    for name, n in (("a1", H), ("h1", H), ("m1", H), ("k1", H), ("a2", H), ("h2", H), ("a3", C)):
        setattr(s, name, s.new(B, n)[1])
    s.aux, s.dloss = s.new(3 * B)[1], s.t(torch.full((B,), 1.0 / B, device="cuda"))
    s.loss_t, s.loss = s.new(B)
    s.d = Slab(s, {"a1": (B, H), "h1": (B, H), "k1": (B, H), "a2": (B, H), "h2": (B, H), "a3": (B, C)})
    s.sq, s.scale, s.norm = s.new(1)[1], s.new(1)[1], s.new(1)[1]
    s.dev.reset_rng(seed & 0x7FFFFFFF or 1)
    s.scratch_level()
    torch.cuda.synchronize()
    return s


def run_classifier(s):
    d = s.dev
    D, H, C, B = (s.case[k] for k in ("D", "H", "C", "B"))
    p, g, q = s.p.dev, s.g.dev, s.d.dev
    d.affine_forward(H, B, D, p["b1"], p["W1"], s.x, s.a1)
    d.unary_forward(lib.OP_TANH, s.a1, s.h1)
    d.dropout_forward(0.2, s.h1, s.m1, s.k1)
    d.affine_forward(H, B, H, p["b2"], p["W2"], s.k1, s.a2)
    d.unary_forward(lib.OP_RECTIFY, s.a2, s.h2)
    d.affine_forward(C, B, H, p["b3"], p["W3"], s.h2, s.a3)
    d.pnls_forward(C, B, s.a3, s.labels, s.aux, s.loss)
    d.zero(s.d.all)
    d.pnls_backward(C, B, s.a3, s.aux, s.dloss, q["a3"])
    d.csum_backward(C, 1, B, q["a3"], 0, g["b3"])
    d.gemm_nt_acc(C, H, B, q["a3"], s.h2, g["W3"])
    d.gemm_tn_acc(H, B, C, p["W3"], q["a3"], q["h2"])
    d.unary_backward(lib.OP_RECTIFY, s.h2, q["h2"], q["a2"])
    d.csum_backward(H, 1, B, q["a2"], 0, g["b2"])
    d.gemm_nt_acc(H, H, B, q["a2"], s.k1, g["W2"])
    d.gemm_tn_acc(H, B, H, p["W2"], q["a2"], q["k1"])
    d.dropout_backward(s.m1, q["k1"], q["h1"])
    d.unary_backward(lib.OP_TANH, s.h1, q["h1"], q["a1"])
    d.csum_backward(H, 1, B, q["a1"], 0, g["b1"])
    d.gemm_nt_acc(H, D, B, q["a1"], s.x, g["W1"])
    n = s.p.all.size
    d.squared_l2norm(n, s.g.all, s.sq)
    d.clip_scale(1, s.sq, 5.0, s.scale, s.norm)
    d.sgd_update_scaled(n, s.p.all, s.g.all, 0.1, s.scale)
    s.scratch_back()
    return [s.loss_t, s.d.views, s.p.views]


def work_classifier(case):
    D, H, C, B = case["D"], case["H"], case["C"], case["B"]
    w = D * H + H * H + H * C
    return {"bytes": 4.0 * (2 * (w + 2 * H + C) + B * (D + 5 * H + 2 * C)), "flops": 2.0 * B * (3 * w - D * H)}


# ---------------------------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------------------------
_KINDS = {
    "train": (prepare_train, run_train, work_train),
    "score": (prepare_score, run_score, work_score),
    "decode": (prepare_decode, run_decode, work_decode),
    "cell": (prepare_cell, run_cell, work_cell),
    "elementwise": (prepare_elementwise, run_elementwise, work_elementwise),
    "layer_norm": (prepare_layer_norm, run_layer_norm, work_layer_norm),
    "lookup": (prepare_lookup, run_lookup, work_lookup),
    "pnls": (prepare_pnls, run_pnls, work_pnls),
    "attention": (prepare_attention, run_attention, work_attention),
    "classifier": (prepare_classifier, run_classifier, work_classifier),
}


def listed():
    return [
        # the baseline's language model, a training step on the fused path: the largest work this package is given
        {"name": "lm_train", "kind": "train", "path": "fused", "V": 10000, "E": 256, "H": 1024, "L": 2, "B": 128, "T": 35,
         "dropout": 0.0},
        # a medium model as an unchanged graph executor drives it, node by node, with dropout; off the 128 grid
        {"name": "lm_train_nodes", "kind": "train", "path": "nodes", "V": 10000, "E": 650, "H": 650, "L": 2, "B": 20,
         "T": 35, "dropout": 0.5},
        # perplexity of held-out sentences: forward only, a batch of ordinary size
        {"name": "lm_score", "kind": "score", "V": 10000, "E": 256, "H": 512, "L": 2, "B": 64, "T": 35},
        # sampling a sentence: one token at batch 1, where latency and launches count
        {"name": "decode_1", "kind": "decode", "V": 10000, "E": 256, "H": 1024, "L": 2, "B": 1},
        # beam or batched generation
        {"name": "decode_32", "kind": "decode", "V": 10000, "E": 256, "H": 1024, "L": 2, "B": 32},
        # the baseline's single cell
        {"name": "cell", "kind": "cell", "I": 128, "H": 256, "B": 32},
        # the baseline's elementwise and reduction sweep
        {"name": "elementwise", "kind": "elementwise", "n": 65536, "bd": 64},
        # the baseline's LayerNorm
        {"name": "layer_norm", "kind": "layer_norm", "n": 1024, "bd": 4096},
        # the baseline's embedding: batch 256 x 64 tokens
        {"name": "lookup", "kind": "lookup", "V": 50000, "D": 512, "n": 16384},
        # the baseline's output loss
        {"name": "pnls", "kind": "pnls", "V": 50000, "B": 512},
        # attention of a translation decoder's timestep over a batch
        {"name": "attention", "kind": "attention", "H": 1024, "T": 35, "B": 128},
        # a classifier's or tagger's step over a minibatch
        {"name": "classifier", "kind": "classifier", "D": 784, "H": 1024, "C": 50, "B": 512},
    ]


def _log(rng, lo, hi, grid=1):
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / grid)) * grid
    return max(lo, min(hi, v))


def _size(rng, lo, hi):
    """A layer's width: often a round number, now and then any."""
    return _log(rng, lo, hi, rng.choice((1, 2, 4, 32, 128)))


def draw(rng):
    kind = rng.choice(sorted(_KINDS))
    if kind == "train":
        path = rng.choice(("fused", "nodes"))
        H = _size(rng, 128, 1024)
        return {"kind": kind, "path": path, "V": _log(rng, 1000, 10000), "E": _size(rng, 64, 256) if path == "fused" else H,
                "H": H, "L": rng.choice((1, 2)), "B": _log(rng, 4, 128), "T": rng.randint(8, 35),
                "dropout": rng.choice((0.0, 0.5))}
    if kind == "score":
        return {"kind": kind, "V": _log(rng, 1000, 10000), "E": _size(rng, 64, 512), "H": _size(rng, 128, 1024),
                "L": rng.choice((1, 2)), "B": _log(rng, 1, 128), "T": rng.randint(5, 35)}
    if kind == "decode":
        return {"kind": kind, "V": _log(rng, 1000, 50000), "E": _size(rng, 64, 512), "H": _size(rng, 128, 1024),
                "L": rng.choice((1, 2)), "B": _log(rng, 1, 64)}
    if kind == "cell":
        return {"kind": kind, "I": _size(rng, 32, 1024), "H": _size(rng, 32, 1024), "B": _log(rng, 1, 256)}
    if kind == "elementwise":
        bd = _log(rng, 1, 1024)
        return {"kind": kind, "n": _log(rng, 64, (1 << 22) // bd), "bd": bd}
    if kind == "layer_norm":
        n = _size(rng, 32, 4096)
        return {"kind": kind, "n": n, "bd": _log(rng, 1, (1 << 22) // n)}
    if kind == "lookup":
        D = _size(rng, 32, 1024)
        return {"kind": kind, "V": _log(rng, 1000, 50000), "D": D, "n": _log(rng, 16, min(65536, (1 << 23) // D))}
    if kind == "pnls":
        V = _log(rng, 1000, 50000)
        return {"kind": kind, "V": V, "B": _log(rng, 1, 25600000 // V)}
    if kind == "attention":
        return {"kind": kind, "H": _size(rng, 64, 1024), "T": _log(rng, 5, 35), "B": _log(rng, 1, 128)}
    return {"kind": kind, "D": _size(rng, 64, 1024), "H": _size(rng, 64, 1024), "C": _log(rng, 5, 100),
            "B": _log(rng, 16, 1024)}


def prepare(case, seed):
    return _KINDS[case["kind"]][0](case, seed)


def run(state):
    return _KINDS[state.case["kind"]][1](state)


def work(case):
    return _KINDS[case["kind"]][2](case)


# About four times the largest distance from the same computation in 64 bits over the listed cases and sixty drawn ones.
_TOLERANCE = {
    "train": {"rel": 4e-6, "max": 1e-4},
    "score": {"rel": 2e-6, "max": 4e-5},
    "decode": {"rel": 1e-6, "max": 2e-5},
    "cell": {"rel": 1e-6, "max": 2e-5},
    "elementwise": {"rel": 5e-7, "max": 2e-5},
    "layer_norm": {"rel": 1e-6, "max": 1e-5},
    "lookup": {"rel": 1e-7, "max": 1e-5},
    "pnls": {"rel": 5e-7, "max": 1e-5},
    "attention": {"rel": 2e-6, "max": 2e-4},
    "classifier": {"rel": 2e-6, "max": 2e-5},
}


def tolerance(case):
    return dict(_TOLERANCE[case["kind"]])
