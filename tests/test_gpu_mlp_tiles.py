"""The warm-start network at the edges of its kernels' tiles: the forward pass
around the 32 contacts of a wave, the gradients around the 128 of a workgroup
and past one tile per workgroup, against 64-bit torch with the network's own
bf16 activations.

Tolerance: products are exact and added in FP32, so sums of up to a few hundred
terms are within 1e-5 of the norm; a hidden sum next to a bf16 rounding midpoint
may round the other way (2^-8 of one of 64 activations, in about 1 row of 4,000
times 128 sums), hence 1e-3 for the gradient norm of few rows and 3e-2 for any
output.  A wrong lane layout or split gives errors of the order of 1."""
import numpy as np
import pytest

from experiments_amd import _lib as L
from experiments_amd.warmstart import Mlp

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def reference(x, t, w16, bias):
    w = torch.from_numpy((w16.astype(np.int32) << 16)).view(torch.float32).double()
    b = torch.from_numpy(bias).double()
    w1, w2, w3 = w[:1024].view(64, 16), w[1024:5120].view(64, 64), w[5120:].view(3, 64)
    r16 = lambda v: v.float().bfloat16().double()  # noqa: E731
    x = r16(x)
    a1 = (x @ w1.T + b[:64]).relu()
    a2 = (r16(a1) @ w2.T + b[64:128]).relu()
    y = r16(a2) @ w3.T + b[128:]
    e = y - t.double()
    dy = 2.0 * e / (3.0 * len(x))
    d2 = (dy @ w3) * (a2 > 0)
    d1 = (d2 @ w2) * (a1 > 0)
    g = torch.cat([(d1.T @ x).reshape(-1), (d2.T @ r16(a1)).reshape(-1), (dy.T @ r16(a2)).reshape(-1),
                   d1.sum(0), d2.sum(0), dy.sum(0)])
    return y, g, float((e * e).mean())


@pytest.mark.parametrize("n", [1, 16, 17, 31, 32, 33, 127, 128, 129, 128 * 256 - 1, 128 * 256 + 1, 98309])
def test_tiles(n):
    gen = torch.Generator().manual_seed(n)
    x = torch.randn((n, 16), generator=gen)
    t = torch.randn((n, 3), generator=gen)
    m = Mlp(seed=7)
    w, _ = m.get_weights()
    bias = np.random.default_rng(n).uniform(-0.2, 0.2, L.MLP_NB).astype(np.float32)
    m.set_weights(w, bias)
    ry, rg, rloss = reference(x, t, w, bias)
    y = m.forward(x.cuda()).cpu().double()
    assert float(((y - ry).abs() / (1 + ry.abs())).max()) <= 3e-2
    assert float((y - ry).norm() / ry.norm()) <= 1e-3
    g, loss = m.gradients(x.cuda(), t.cuda())
    g = g.cpu().double()
    for lo, hi in ((0, 1024), (1024, 5120), (5120, 5312), (5312, 5376), (5376, 5440), (5440, 5443)):
        assert float((g[lo:hi] - rg[lo:hi]).norm() / rg[lo:hi].norm()) <= 1e-3, (lo, hi)
    assert abs(loss - rloss) <= 1e-4 * rloss
    m.close()
