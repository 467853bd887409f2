"""Pair searches at the edges of their kernels: every body's range length around
the sorting networks (8, 16, 32 pairs and one more), sweeps of a few AABBs
around a wave's 8 and a workgroup's 32 owners and 64 candidates, sets so dense
that a workgroup's pairs do not fit its record and are swept again, and bounds
that are infinite, NaN, of zero extent or signed zeros.  Integer results, equal
to the brute-force overlap set."""
import ctypes

import numpy as np
import pytest

from experiments_amd import _lib as L

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def brute(mn, mx):
    a = np.ones((len(mn), len(mn)), bool)
    for k in range(3):
        a &= (mn[:, None, k] <= mx[None, :, k]) & (mn[None, :, k] <= mx[:, None, k])
    x, y = np.nonzero(np.tril(a, -1))
    return np.stack([x, y], 1).astype(np.int32)


def search(kind, mn, mx, cap, large=None, axis=0):
    n = len(mn)
    d = [torch.from_numpy(np.ascontiguousarray(np.pad(v.astype(np.float32), ((0, 0), (0, 1))))).cuda()
         for v in (mn, mx)]
    pairs = torch.zeros((cap, 2), dtype=torch.int32, device="cuda")
    num = torch.zeros(1, dtype=torch.int32, device="cuda")
    lg = None if large is None else torch.from_numpy(large.astype(np.int32)).cuda()
    h = ctypes.c_void_p()
    if kind == "sap":
        L.call("mi_rb_sap_create", ctypes.byref(L.SapDesc(axis, cap)), n, ctypes.byref(h))
    else:
        L.call("mi_rb_grid_create", ctypes.byref(L.GridDesc(2.0, (ctypes.c_int * 3)(16, 16, 16), cap, 1, 4)),
               n, ctypes.byref(h))
    vp = lambda t: None if t is None else ctypes.c_void_p(t.data_ptr())  # noqa: E731
    for _ in range(2):  # a handle is used again
        L.call("mi_rb_%s_find_pairs" % kind, h, vp(d[0]), vp(d[1]), vp(lg), n, vp(pairs), vp(num), None)
    torch.cuda.synchronize()
    getattr(L.lib(), "mi_rb_%s_destroy" % kind)(h)
    return pairs[:int(num.cpu()[0])].cpu().numpy()


@pytest.mark.parametrize("kind", ["sap", "grid"])
@pytest.mark.parametrize("n", [2, 9, 17, 33, 34, 65, 300])
def test_every_range_length(kind, n):
    """All overlap: body x has x pairs, in an order the search must restore."""
    rng = np.random.default_rng(n)
    c = rng.uniform(-0.3, 0.3, (n, 3))
    mn, mx = (c - 0.5).astype(np.float32), (c + 0.5).astype(np.float32)
    assert np.array_equal(search(kind, mn, mx, n * n), brute(mn, mx))


@pytest.mark.parametrize("n", [1, 7, 8, 9, 31, 32, 33, 63, 64, 65, 71, 72, 73, 129, 1000])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_sweep_edges(n, axis):
    rng = np.random.default_rng(n + axis)
    c = rng.uniform(0, 0.9 * n ** (1 / 3), (n, 3))
    mn, mx = (c - 0.5).astype(np.float32), (c + 0.5).astype(np.float32)
    mn[::5] = np.round(mn[::5])  # equal mins and touching faces
    large = np.zeros(n, int)
    large[n // 2::37] = 1
    assert np.array_equal(search("sap", mn, mx, 64 * n + 64, large, axis), brute(mn, mx))


def test_sweep_of_odd_bounds():
    rng = np.random.default_rng(3)
    c = rng.uniform(-4, 4, (400, 3))
    mn, mx = (c - 0.6).astype(np.float32), (c + 0.6).astype(np.float32)
    mn[3], mx[3] = -1e30, 1e30
    mn[4], mx[4] = -np.inf, np.inf
    mx[5, 0] = np.inf
    mn[6], mx[7] = np.nan, np.nan
    mn[8, 0] = -np.float32(np.nan)
    mx[9:20] = mn[9:20]
    mn[20], mx[20] = 0.0, 0.0
    mn[21], mx[21] = -0.0, -0.0
    mn[22], mx[22] = mx[22].copy(), mn[22].copy()  # inside out: overlaps what spans both
    assert np.array_equal(search("sap", mn, mx, 1 << 17), brute(mn, mx))
