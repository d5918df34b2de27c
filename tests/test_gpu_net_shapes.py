"""The net's kernels at the edges of their tiles (strips of 16 and 32
columns, segments of 8 rows, images smaller than either) against a numpy
restatement with the same BF16 rounding points and FP64 sums.  Both round
the same values to BF16; where their FP32 / FP64 sums fall on different
sides of a rounding boundary (about one value in 10^4) one element moves by
2^-8, so a block of values agrees to well under 2e-3 of its norm."""
import numpy as np
import pytest

from nutrlan_amd import learned
from test_gpu_net import bf16, unpack

pytestmark = pytest.mark.gpu
TOL = 2e-3


def b16(a):
    return bf16(a.astype(np.float32)).astype(np.float64)


def tap(a, t, sign=1):
    """a at pixel + sign * (dy, dx) of tap t."""
    return np.roll(a, (-sign * (t // 3 - 1), -sign * (t % 3 - 1)), (1, 2))


def restated(p, x, tg):
    w1, b1, w2, b2, w3, b3, w4, b4 = [v.astype(np.float64) for v in unpack(p)]
    w1, w2, w3, w4 = b16(w1), b16(w2), b16(w3), b16(w4)
    xr = b16(x)
    a1 = b16(np.maximum(sum(tap(xr, t)[..., None] * w1[:, t] for t in range(9)) + b1, 0))
    a2 = b16(np.maximum(sum(tap(a1, t) @ w2[:, t].T for t in range(9)) + b2, 0))
    a3 = b16(np.maximum(sum(tap(a2, t) @ w3[:, t].T for t in range(9)) + b3, 0))
    o = (sum(tap(a3, t) @ w4[t] for t in range(9)) + b4[0]).astype(np.float32).astype(np.float64)
    ot, oo, tt = [(u * v).sum((1, 2), keepdims=True) for u, v in ((o, tg), (o, o), (tg, tg))]
    c = ot * ot / (oo * tt)
    do = (2.0 / len(x) * (c * o / oo - ot * tg / (oo * tt))).astype(np.float32).astype(np.float64)
    dr = b16(do)
    d3 = b16((a3 > 0) * sum(tap(dr, t, -1)[..., None] * w4[t] for t in range(9)))
    d2 = b16((a2 > 0) * sum(tap(d3, t, -1) @ w3[:, t] for t in range(9)))
    d1 = b16((a1 > 0) * sum(tap(d2, t, -1) @ w2[:, t] for t in range(9)))

    def dw(dy, a):  # [co][t][ci]
        return np.stack([np.einsum("byxo,byxi->oi", dy, tap(a, t)) for t in range(9)], 1)

    g = [np.stack([np.einsum("byxo,byx->o", d1, tap(xr, t)) for t in range(9)], 1), d1.sum((0, 1, 2)),
         dw(d2, a1), d2.sum((0, 1, 2)), dw(d3, a2), d3.sum((0, 1, 2)),
         np.stack([np.einsum("byx,byxi->i", dr, tap(a3, t)) for t in range(9)], 0), do.sum()]
    return o, (1 - c).mean(), g


@pytest.mark.parametrize("shape", [(2, 3, 3), (1, 5, 16), (3, 8, 17), (2, 9, 31), (1, 16, 32), (2, 17, 33),
                                   (1, 7, 65), (5, 40, 4), (90, 12, 40)])
def test_forward_and_gradients(gpu_lib, shape):
    net = learned.Net(seed=21)
    rng = np.random.default_rng(22)
    x = rng.uniform(-1, 1, shape).astype(np.float32)
    t = np.abs(rng.standard_normal(shape)).astype(np.float32)
    print(f"net shape {shape}", flush=True)
    o, loss, blocks = restated(net.params(), x, t.astype(np.float64))
    y = net.forward(x)
    assert np.linalg.norm(y - o) <= TOL * np.linalg.norm(o)
    got, g = net.loss_grad(x, t)
    assert abs(got - loss) <= TOL * loss
    at = 0
    for b in blocks:
        b = np.atleast_1d(b).ravel()
        d = g[at:at + b.size]
        at += b.size
        # the last bias sums gradients that nearly cancel: against their size
        ref = max(np.linalg.norm(b), 1e-2 * np.abs(blocks[6]).max())
        assert np.linalg.norm(d - b) <= TOL * ref, (at, np.linalg.norm(d - b) / ref)
    net.close()


@pytest.mark.parametrize("shape", [(130, 17, 33), (90, 33, 18), (33, 30, 47)])
def test_more_waves(gpu_lib, shape):
    """Batches of more waves than SIMDs, which walk 8 or 4 rows each (those
    above walk 2 or 4); ragged in both directions."""
    test_forward_and_gradients(gpu_lib, shape)


@pytest.mark.parametrize("shape", [(1, 4, 3), (5, 9, 3), (6, 17, 3), (16, 5, 4), (7, 6, 5), (9, 3, 6), (4, 11, 7),
                                   (3, 8, 8), (66, 3, 8), (2, 5, 9)])
def test_narrow_images(gpu_lib, shape):
    """Images that share a strip: each one's output is that of the image
    alone."""
    test_forward_and_gradients(gpu_lib, shape)
    net = learned.Net(seed=21)
    x = np.random.default_rng(23).uniform(-1, 1, shape).astype(np.float32)
    y = net.forward(x)
    for i in range(len(x)):
        assert np.array_equal(net.forward(x[i:i + 1])[0], y[i]), i
    net.close()


@pytest.mark.parametrize("shape", [(1, 8, 8), (1, 20, 20), (6, 6, 5), (3, 50, 71), (1, 64, 64), (40, 64, 33)])
def test_last_bias_gradient(gpu_lib, shape):
    """The last layer's bias sums loss gradients that nearly cancel, in FP64:
    the result is rounded once (2^-24), and one in 10^3 of the summands may
    differ by a rounding from those formed here."""
    for k in range(4):
        net = learned.load_net()
        rng = np.random.default_rng(100 * shape[0] + k)
        x = rng.uniform(-1, 1, shape).astype(np.float32)
        t = np.abs(rng.standard_normal(shape)).astype(np.float32)
        o, tg = net.forward(x).astype(np.float64), t.astype(np.float64)
        ot, oo, tt = [(u * v).sum((1, 2), keepdims=True) for u, v in ((o, tg), (o, o), (tg, tg))]
        c = ot * ot / (oo * tt)
        do = (2.0 / len(x) * (c * o / oo - ot * tg / (oo * tt))).astype(np.float32).astype(np.float64)
        g = net.loss_grad(x, t)[1][-1]
        assert abs(g - do.sum()) <= 2.0 ** -24 * (abs(do.sum()) + 1e-3 * np.abs(do).sum()), (k, g, do.sum())
        net.close()
