"""All timesteps of an LSTM layer in one launch (dyhip_lstm_sequence_forward / _backward) against fp64, at the edges of its
tiles, with tiles taken over from blocks that are not there, and beside another launch of itself."""
import numpy as np
import pytest

from dynet_amd import DyhipError

pytestmark = pytest.mark.gpu

# H 16 and 32: a row tile; B 16 and 32: a column tile; H 1024: the largest; (512, 64), (1024, 128): every CU or half of them
SIZES = [(1, 1, 3), (15, 16, 2), (16, 17, 3), (17, 33, 4), (127, 5, 3), (128, 32, 4), (200, 33, 1), (257, 40, 3), (8, 300, 2),
         (512, 64, 4), (650, 20, 4), (513, 70, 3), (1000, 100, 2), (1024, 1, 3), (1024, 128, 3)]


def _f(a):
    return np.ascontiguousarray(a, dtype=np.float32)


def _d(a):
    return np.asarray(a, dtype=np.float64)


def _sigmoid(x):
    with np.errstate(over="ignore"):
        return 1.0 / (1.0 + np.exp(-x))


class Case:
    def __init__(self, H, B, T, mask, seed=0):
        rng = np.random.default_rng(seed + H * 7 + B)
        s = np.sqrt(6.0 / (5 * H))
        self.H, self.B, self.T = H, B, T
        self.Wh = _f(rng.uniform(-s, s, (H, 4 * H)))  # numpy order of a column-major 4H x H matrix
        self.x = _f(rng.normal(0, 0.5, (T, B, 4 * H)))
        self.b = _f(rng.normal(0, 0.1, 4 * H))
        self.dh = _f(rng.normal(0, 1, (T, B, H)))
        self.mask = _f((rng.random((B, H)) < 0.5) * 2.0) if mask else None

    def forward(self):
        H, m = self.H, 1.0 if self.mask is None else _d(self.mask)
        h, c = np.zeros((self.B, H)), np.zeros((self.B, H))
        gates, cs, hs = [], [], []
        for t in range(self.T):
            pre = _d(self.x[t]) + self.b
            if t > 0:
                pre = pre + (h * m) @ _d(self.Wh)
            i, f, o = (_sigmoid(pre[:, k * H:(k + 1) * H] + (k == 1)) for k in range(3))
            g = np.tanh(pre[:, 3 * H:])
            c = i * g + f * c if t > 0 else i * g
            h = o * np.tanh(c)
            gates.append(np.concatenate([i, f, o, g], 1)), cs.append(c), hs.append(h)
        return np.stack(gates), np.stack(cs), np.stack(hs)

    def backward(self, gates, cs):
        H, m = self.H, 1.0 if self.mask is None else _d(self.mask)
        out, dc, dpre = [None] * self.T, 0.0, None
        for t in reversed(range(self.T)):
            i, f, o, g = (_d(gates[t][:, k * H:(k + 1) * H]) for k in range(4))
            dh = _d(self.dh[t])
            if dpre is not None:
                dh = dh + (dpre @ _d(self.Wh).T) * m
            th = np.tanh(_d(cs[t]))
            dcv = dc + dh * o * (1 - th * th)
            df = dcv * _d(cs[t - 1]) * f * (1 - f) if t > 0 else 0.0 * f * (1 - f)
            dpre = np.concatenate([dcv * g * i * (1 - i), df, dh * th * o * (1 - o), dcv * i * (1 - g * g)], 1)
            dc = dcv * f
            out[t] = dpre
        return np.stack(out)

    def place(self, dev):
        t = dev.tensor
        self.t = {n: t(getattr(self, n)) for n in ("Wh", "x", "b", "dh")}
        self.t["mask"] = None if self.mask is None else t(self.mask)
        T, B, H = self.T, self.B, self.H
        self.gates, self.c, self.h, self.dpre = (dev.empty((T, B, n)) for n in (4 * H, H, H, 4 * H))
        nbytes = dev.lstm_sequence_workspace(H, B, T)
        assert nbytes > 0
        self.ws = dev.workspace(nbytes)
        return self

    def run_forward(self, q):
        q.lstm_sequence_forward(self.H, self.B, self.T, self.t["Wh"], self.t["x"], self.t["b"], self.gates, self.c, self.h,
                                *self.ws, mask_h=self.t["mask"])

    def run_backward(self, q, gates, c):
        q.lstm_sequence_backward(self.H, self.B, self.T, self.t["Wh"], gates, c, self.t["dh"], self.dpre, *self.ws,
                                 mask_h=self.t["mask"])


@pytest.mark.parametrize("mask", [False, True])
@pytest.mark.parametrize("H,B,T", SIZES)
def test_sequence_matches_fp64(dev, H, B, T, mask):
    k = Case(H, B, T, mask).place(dev)
    k.run_forward(dev)
    gates, c, h = k.forward()
    # a pre-activation is a sum of up to 1024 products below 0.1 in magnitude and near 1: a few 1e-7; its error passes
    # through activations of slope <= 1 and T <= 4 timesteps
    for got, ref in ((k.gates, gates), (k.c, c), (k.h, h)):
        assert np.max(np.abs(got.numpy() - ref)) < 2e-6
    g32, c32 = dev.tensor(_f(gates)), dev.tensor(_f(c))
    k.run_backward(dev, g32, c32)
    ref = k.backward(_f(gates), _f(c))
    # 4096 products a sum; T sums one into the other
    assert np.linalg.norm(k.dpre.numpy() - ref) <= 1e-6 * np.linalg.norm(ref)
    assert np.max(np.abs(k.dpre.numpy() - ref)) <= 1e-5 * max(1.0, np.max(np.abs(ref)))


@pytest.mark.parametrize("H,B,T,blocks", [(40, 16, 4, 1), (300, 16, 5, 7), (300, 30, 3, 20), (1000, 16, 3, 40)])
def test_sequence_without_some_of_its_blocks(dev, H, B, T, blocks):
    """Blocks that do not find a place on the GPU: the others take their tiles; the same bits."""
    k = Case(H, B, T, True).place(dev)
    k.run_forward(dev)
    want = [t.numpy() for t in (k.gates, k.c, k.h)]
    k.run_backward(dev, k.gates, k.c)
    want.append(k.dpre.numpy())
    gates, c = dev.tensor(want[0]), dev.tensor(want[1])
    for t in (k.gates, k.c, k.h, k.dpre):
        dev.zero(t)
    dev.set_sequence_blocks(blocks)
    try:
        k.run_forward(dev)
        if B <= 16:  # one column tile backward: the blocks that are there can see what is missing
            k.run_backward(dev, gates, c)
    finally:
        dev.set_sequence_blocks(0)
    for t, w in list(zip((k.gates, k.c, k.h, k.dpre), want))[:4 if B <= 16 else 3]:
        np.testing.assert_array_equal(t.numpy(), w)


def test_sequences_on_two_queues_at_once(dev):
    """Each launch wants every CU: whichever blocks run, both end, with the same bits as alone."""
    q = dev.fork()
    try:
        a, b = Case(1024, 128, 6, False, 1).place(dev), Case(1024, 128, 6, True, 2).place(dev)
        want = []
        for k in (a, b):
            k.run_forward(dev)
            k.run_backward(dev, k.gates, k.c)
            want.append([t.numpy() for t in (k.gates, k.h, k.dpre)])
        dev.sync()
        for _ in range(6):
            a.run_forward(dev)
            b.run_forward(q)
            a.run_backward(dev, a.gates, a.c)
            b.run_backward(q, b.gates, b.c)
            dev.sync()
            q.sync()
            for k, w in zip((a, b), want):
                for t, v in zip((k.gates, k.h, k.dpre), w):
                    np.testing.assert_array_equal(t.numpy(), v)
    finally:
        q.close()


def test_sequence_replayed_from_a_graph(dev):
    k = Case(300, 40, 5, True).place(dev)
    k.run_forward(dev)
    want = k.h.numpy()
    dev.graph_begin()
    k.run_forward(dev)
    k.run_backward(dev, k.gates, k.c)
    g = dev.graph_end()
    for _ in range(3):
        dev.zero(k.h)
        g.launch()
        np.testing.assert_array_equal(k.h.numpy(), want)
    g.destroy()


def test_sequence_keeps_infinities_nans_and_small_values(dev):
    k = Case(70, 20, 4, False)
    k.Wh[3, 40] = np.inf   # one gate saturates from the second timestep on
    k.Wh[5, 200] = 1e38    # a sum far above 2^96
    k.x[0, 7, :] = np.nan  # one sentence is lost
    k.dh[:, 11, :] *= np.float32(2.0 ** -125)
    k.dh[3, 13, 2] = np.inf
    k.place(dev)
    k.run_forward(dev)
    with np.errstate(invalid="ignore", over="ignore"):
        gates, c, h = k.forward()
    others = [b for b in range(20) if b != 7]  # (the logistic of a NaN is 1, as in the reference)
    np.testing.assert_allclose(k.gates.numpy()[:, others], gates[:, others], rtol=0, atol=2e-6)
    np.testing.assert_allclose(k.h.numpy(), h, rtol=0, atol=2e-6)
    k.Wh[3, 40], k.Wh[5, 200] = 0.1, 0.1
    k.place(dev)
    g32, c32 = _f(gates), _f(c)
    k.run_backward(dev, dev.tensor(g32), dev.tensor(c32))
    with np.errstate(invalid="ignore", over="ignore"):
        ref = k.backward(g32, c32)
    got = k.dpre.numpy()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(ref))
    small = ref[:, 11]
    assert np.linalg.norm(got[:, 11].astype(np.float64) - small) <= 2e-6 * np.linalg.norm(small) + 2.0 ** -149 * small.size
    rest = [b for b in range(20) if b not in (7, 11, 13)]
    assert np.linalg.norm(got[:, rest] - ref[:, rest]) <= 1e-6 * np.linalg.norm(ref[:, rest])


@pytest.mark.parametrize("power", [90, 110, 111, 118])
def test_sequence_keeps_large_gradients(dev, power):
    """Gradients up to fp32's range reach the timesteps before theirs: nothing counts as infinite that is not."""
    k = Case(70, 20, 4, True)
    k.dh[:, 11, :] *= np.float32(2.0 ** power)
    k.dh[3, 13, 2] = np.float32(2.0 ** 120)
    gates, c, _ = k.forward()
    g32, c32 = _f(gates), _f(c)
    ref = k.backward(g32, c32)
    assert np.max(np.abs(ref)) < 2.0 ** 124
    k.place(dev)
    k.run_backward(dev, dev.tensor(g32), dev.tensor(c32))
    got = _d(k.dpre.numpy())
    for b in range(20):
        for t in range(4):
            assert np.linalg.norm(got[t, b] - ref[t, b]) <= 2e-6 * np.linalg.norm(ref[:, b])


def test_sequence_reports_a_wait_that_gave_up_and_refuses_what_it_cannot_do(dev):
    k = Case(300, 40, 30, False).place(dev)
    k.run_forward(dev)
    want = k.h.numpy()
    dev.set_gemm_handoff(0, True)  # a wait that is not over at the first look gives up
    try:
        k.run_forward(dev)
        with pytest.raises(DyhipError, match="gave up"):
            dev.sync()
    finally:
        dev.set_gemm_handoff()
    k.run_forward(dev)
    np.testing.assert_array_equal(k.h.numpy(), want)
    assert dev.lstm_sequence_workspace(1025, 4, 3) == 0 and dev.lstm_sequence_workspace(1024, 200, 3) == 0
    ws, nbytes = k.ws
    for bad in ((ws, 1000), (ws + 4, nbytes), (None, 0)):
        k.ws = bad
        with pytest.raises(DyhipError):
            k.run_forward(dev)
