"""The exclusive scan at the edges of its tiles (4,096 words, moved 16 bytes a
lane when the arrays are aligned), with arrays that start off a 16-byte
boundary, in place, and with a sum that wraps."""
import ctypes

import numpy as np
import pytest

from experiments_amd import _lib as L

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 4, 5, 4095, 4096, 4097, 8192, 12289, 64 * 4096 + 1, 300001])
@pytest.mark.parametrize("off_in,off_out", [(0, 0), (1, 0), (0, 3), (2, 2)])
def test_exclusive_scan(n, off_in, off_out):
    rng = np.random.default_rng(n)
    x = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    din = torch.zeros(n + 4, dtype=torch.int32, device="cuda")
    din[off_in:off_in + n] = torch.from_numpy(x.view(np.int32)).cuda()
    dout = torch.full((n + 8,), -7, dtype=torch.int32, device="cuda")
    tot = torch.zeros(1, dtype=torch.int32, device="cuda")
    h = ctypes.c_void_p()
    L.call("mi_rb_radix_sort_create", n, ctypes.byref(h))
    ref = np.concatenate([[0], np.cumsum(x, dtype=np.uint32)]).astype(np.uint32)
    at = lambda t, o: ctypes.c_void_p(t.data_ptr() + 4 * o)  # noqa: E731
    for _ in range(2):
        L.call("mi_rb_exclusive_scan_u32", h, at(din, off_in), at(dout, off_out), n, at(tot, 0), None)
    torch.cuda.synchronize()
    got = dout.cpu().numpy().view(np.uint32)
    assert np.array_equal(got[off_out:off_out + n], ref[:-1])
    assert np.all(got[:off_out] == 0xFFFFFFF9) and np.all(got[off_out + n:] == 0xFFFFFFF9)
    assert int(tot.cpu().numpy().view(np.uint32)[0]) == int(ref[-1])
    L.call("mi_rb_exclusive_scan_u32", h, at(din, off_in), at(din, off_in), n, None, None)
    torch.cuda.synchronize()
    assert np.array_equal(din.cpu().numpy().view(np.uint32)[off_in:off_in + n], ref[:-1])
    L.lib().mi_rb_radix_sort_destroy(h)
