"""The precision of the network's backward pass: each FP32 delta enters the
products as three bf16 terms, whose sum is the delta, so a gradient is as exact
as FP32 sums of FP32 deltas.

Small integers as inputs, weights and biases make every hidden sum exact in any
order (nothing rounds the other way, unlike in the tile tests), and targets of
full mantissa give full deltas.  Tolerance, per parameter block and of its norm:
about 16 roundings meet in a sum here (3 products' sums a wave, 4 waves, 2
workgroups, the products' own), 2^-24 each and of either sign: 2.4e-7; three
times that is allowed.  Two terms instead of three are off by 2^-17 of a delta
at most and by 1.6e-6 to 2.6e-6 of a block's norm, as the first test shows."""
import numpy as np
import pytest

from experiments_amd.warmstart import Mlp

torch = pytest.importorskip("torch")

BLOCKS = ((0, 1024), (1024, 5120), (5120, 5312), (5312, 5376), (5376, 5440), (5440, 5443))
TOLERANCE = 7.2e-7


def r16(v):
    return torch.from_numpy(np.ascontiguousarray(v)).float().bfloat16().double().numpy()


def terms(v, k):
    """The sum of the first k bf16 terms of v."""
    v, s = v.astype(np.float32), 0.0
    for _ in range(k):
        t = r16(v).astype(np.float32)
        s, v = s + t.astype(np.float64), v - t
    return s


def problem(n):
    rng = np.random.default_rng(n)
    w = np.zeros(5312)
    w[:1024] = rng.integers(-1, 2, 1024)
    w[1024:5120] = rng.integers(-1, 2, 4096) * (rng.random(4096) < 0.25)
    w[5120:] = rng.choice([-1.0, 1.0], 192)
    b = np.zeros(131)
    b[:64] = rng.integers(-2, 3, 64)
    b[64:128] = rng.integers(-4, 5, 64)
    x = rng.integers(-2, 3, (n, 16)).astype(np.float64)
    w1, w2, w3 = w[:1024].reshape(64, 16), w[1024:5120].reshape(64, 64), w[5120:].reshape(3, 64)
    a1 = np.maximum(x @ w1.T + b[:64], 0.0)
    a2 = np.maximum(r16(a1) @ w2.T + b[64:128], 0.0)
    b[128:] = -np.round((r16(a2) @ w3.T).mean(0))  # errors of either sign
    y = r16(a2) @ w3.T + b[128:]
    t = (100.0 * rng.normal(size=(n, 3))).astype(np.float32)
    return x, t, w, b, (w2, w3, a1, a2, y)


def gradients(n, used=None):
    """In 64 bits; with `used`, FP32 deltas that enter the four products (dW1,
    dW2, layer 1's deltas, dW3) as so many bf16 terms."""
    x, t, _, _, (w2, w3, a1, a2, y) = problem(n)
    f32 = (lambda v: v) if used is None else (lambda v: v.astype(np.float32).astype(np.float64))
    part = (lambda v, i: v) if used is None else (lambda v, i: terms(v, used[i]))
    dy = f32(2.0 * f32(y - t.astype(np.float64)) / (3.0 * n))
    d2 = f32(dy @ w3) * (a2 > 0)
    d1 = f32(part(d2, 2) @ w2) * (a1 > 0)
    g = [part(d1, 0).T @ x, part(d2, 1).T @ r16(a1), part(dy, 3).T @ r16(a2),
         d1.sum(0), d2.sum(0), dy.sum(0)]
    return np.concatenate([v.reshape(-1) for v in g])


def errors(g, ref):
    return [float(np.linalg.norm(g[lo:hi] - ref[lo:hi]) / np.linalg.norm(ref[lo:hi]))
            for lo, hi in BLOCKS]


@pytest.mark.parametrize("n", [33, 64, 128, 160])
def test_two_terms_exceed_the_tolerance(n):
    ref = gradients(n)
    assert max(errors(gradients(n, (3, 3, 3, 3)), ref)) < 0.3 * TOLERANCE
    for product, block in ((0, 0), (1, 1), (2, 0), (2, 3), (3, 2)):
        used = [3, 3, 3, 3]
        used[product] = 2
        assert errors(gradients(n, used), ref)[block] > 2.0 * TOLERANCE, (product, block)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [33, 64, 128, 160])
def test_gradients_are_as_exact_as_fp32(n):
    x, t, w, b, _ = problem(n)
    m = Mlp(seed=1)
    m.set_weights(torch.from_numpy(w).bfloat16().view(torch.int16).numpy().view(np.uint16),
                  b.astype(np.float32))
    g, _ = m.gradients(torch.from_numpy(x).float().cuda(), torch.from_numpy(t).cuda())
    e = errors(g.cpu().double().numpy(), gradients(n))
    assert max(e) <= TOLERANCE, e
    m.close()
