"""The step's pair search: dense clusters whose bodies have from none to over a
hundred overlaps, with room for 1 to 64 a body, in grids of 4 to 64 cells an
axis (wrapped), alone (2 entries a wave) and among so many bodies that 4 or 16
entries share a wave.  A body's pairs are the first ones of a serial search:
stencil cells in z, y, x order, members in sorted order, large bodies last."""
import numpy as np
import pytest

import oracle as O
from experiments_amd import _lib as L
from experiments_amd import scenes
from oracle.step import Snapshot, oracle_broadphase

pytestmark = pytest.mark.gpu


def expected(s, mn, mx, skv, pairs, room):
    """The oracle's pairs, each body's cut to the first `room` found."""
    dims, inv = s.params["dims"], np.float32(s.params["inv_cell"])
    place = np.empty(len(skv), np.int64)
    place[skv[:, 1]] = np.arange(len(skv))
    cell = np.floor((mn[:, :3] + mx[:, :3]) * np.float32(0.5) * inv).astype(np.int64)
    kept, over = [], False
    lists = np.split(pairs, np.nonzero(np.diff(pairs[:, 0]))[0] + 1)
    for p in lists:
        if len(p) > room:
            over = True
            i, j = p[0, 0], p[:, 1]
            d = (cell[j] - cell[i] + 1) % np.array(dims)
            large = np.asarray(s.is_large)[j] != 0
            assert d[~large].max() <= 2
            d[large] = 3
            order = np.lexsort((place[j], d[:, 0], d[:, 1], d[:, 2]))
            p = p[np.sort(order[:room])]
        kept.append(p)
    return np.concatenate(kept), over


@pytest.mark.parametrize("room,dims,others", [
    (room, dims, 0) for room in (1, 20, 63, 64) for dims in ((4, 4, 4), (8, 4, 16), (64, 64, 64))
] + [(20, (64, 64, 64), 131072), (64, (64, 64, 64), 131072)])
def test_first_pairs(room, dims, others):
    rng = np.random.default_rng(room)
    sc = scenes.Scene("cluster", iterations=1)
    sc.shapes = [scenes.cube_points(0.5), scenes.box_points(400.0, 1.0, 400.0)]
    at = np.concatenate([rng.uniform(-1.6, 1.6, (260, 3)), rng.uniform(-4.0, 4.0, (77, 3))])
    if others:
        g = np.arange(others)
        far = np.stack([g % 64, g // 64 % 64, g // 4096], 1) * 2.2 + [8.0, 0.0, 8.0]
        at = np.concatenate([at, far])
    q = rng.normal(size=(len(at), 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    if not others:
        sc.add(0.0, (0.0, -3.0, 0.0), (0.0, 0.0, 0.0, 1.0), 1)
    for a, b in zip(at, q):
        sc.add(1.0, tuple(a), tuple(b), 0)
    w = scenes.build_world(sc, max_pairs_per_body=room, max_pairs=1 << 20, max_contacts=1 << 14,
                           grid_dims=dims)
    s = Snapshot(w)
    w.step_partial(L.STAGE_PAIRS)
    mn, mx, skv, pairs = oracle_broadphase(s)
    per_body = np.bincount(pairs[:, 0])
    assert per_body.max() > 100
    ref, over = expected(s, mn, mx, skv, pairs, room)
    assert np.array_equal(w.pairs(), ref)
    assert over
    assert bool(w.stats()["overflow_flags"] & L.OVERFLOW_BODY_PAIRS) == over
    w.close()


@pytest.mark.parametrize("room", [1, 20, 64])
def test_first_pairs_of_four_entries(room):
    test_first_pairs(room, (64, 64, 64), 16384)


@pytest.mark.parametrize("n", [2, 3, 8191, 8192, 8193, 49151, 49152, 49153])
def test_entries_per_wave(n):
    """Around the body counts at which a wave takes 2, 4 or 16 entries."""
    rng = np.random.default_rng(n)
    side = 1.2 * (n / 10.0) ** 0.5 + 1.0
    sc = scenes.Scene("layer", iterations=1)
    sc.shapes = [scenes.cube_points(0.5)]
    at = rng.uniform(-0.5, 0.5, (n, 3)) * [side, 12.0, side]
    q = rng.normal(size=(n, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    for a, b in zip(at, q):
        sc.add(1.0, tuple(a), tuple(b), 0)
    w = scenes.build_world(sc, max_pairs_per_body=64, max_pairs=1 << 20, max_contacts=1 << 14)
    w.step_partial(L.STAGE_PAIRS)
    assert np.array_equal(w.pairs(), O.find_pairs_brute(*w.aabbs()))
    w.close()


@pytest.mark.parametrize("others", [0, 16384, 49152])  # 2, 4 and 16 entries a wave
@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 2, 2), (1, 2, 8), (2, 8, 1), (8, 1, 2)])
def test_small_grids(dims, others):
    """One or two cells on an axis: a cell that is a neighbour on both sides is
    searched once, and every pair is there once."""
    rng = np.random.default_rng(others + dims[0])
    sc = scenes.Scene("small", iterations=1)
    sc.shapes = [scenes.cube_points(0.5), scenes.box_points(400.0, 1.0, 400.0)]
    at = rng.uniform(-6.0, 6.0, (700, 3))
    if others:
        g = np.arange(others)
        at = np.concatenate([at, np.stack([g % 64, g // 64 % 64, g // 4096], 1) * 2.2 + [8.0, 0.0, 8.0]])
    q = rng.normal(size=(len(at), 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    sc.add(0.0, (0.0, -7.0, 0.0), (0.0, 0.0, 0.0, 1.0), 1)
    for a, b in zip(at, q):
        sc.add(1.0, tuple(a), tuple(b), 0)
    w = scenes.build_world(sc, max_pairs=1 << 18, max_contacts=1 << 14, grid_dims=dims)
    assert tuple(w.params()["dims"]) == dims
    w.step_partial(L.STAGE_PAIRS)
    mn, mx = w.aabbs()
    ref = O.find_pairs_brute(mn, mx)
    assert len(ref) > 700
    assert np.array_equal(w.pairs(), ref)
    assert w.stats()["overflow_flags"] == 0
    w.step(1)
    w.close()


@pytest.mark.parametrize("n,dims", [(1500, (4, 4, 4)), (9000, (64, 64, 64)), (50000, (8, 8, 8))])
@pytest.mark.parametrize("room", [1, 33, 64])
def test_first_pairs_of_crowded_cells(n, dims, room):
    """Cells of more members than a half wave reads at once, most lists full,
    entries next to the grid's edges among them."""
    rng = np.random.default_rng(n)
    sc = scenes.Scene("crowd", iterations=1)
    sc.shapes = [scenes.cube_points(0.5)]
    box = {1500: 6.0, 9000: 9.0, 50000: 14.0}[n]
    for p in rng.uniform(-0.5 * box, 0.5 * box, (n, 3)):
        sc.add(1.0, tuple(p), (0.0, 0.0, 0.0, 1.0), 0)
    w = scenes.build_world(sc, max_pairs_per_body=room, max_pairs=64 * n, max_contacts=1 << 12,
                           grid_dims=dims)
    s = Snapshot(w)
    w.step_partial(L.STAGE_PAIRS)
    ref, over = expected(s, *oracle_broadphase(s), room)
    assert over
    assert np.array_equal(w.pairs(), ref)
    w.close()
