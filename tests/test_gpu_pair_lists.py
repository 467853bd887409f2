"""The narrowphase's pair lists at the edges of their 4,096-pair tiles: n bodies
side by side on a ground, one pair each, of small hulls (cubes), large ones (12
vertices) or a mix, some lifted off.  Every contact is listed once, in pair
order, as the oracle has it."""
import numpy as np
import pytest

import oracle as O
from experiments_amd import _lib as L
from experiments_amd import scenes
from oracle.step import Snapshot, oracle_broadphase, oracle_contacts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 4095, 4096, 4097, 8193])
@pytest.mark.parametrize("large", ["none", "all", "some"])
def test_contact_list(n, large):
    rng = np.random.default_rng(n)
    g = (1 + 5 ** 0.5) / 2
    ico = np.array([(0, a, b * g) for a in (-1, 1) for b in (-1, 1)], np.float32)
    ico = np.concatenate([ico, ico[:, [2, 0, 1]], ico[:, [1, 2, 0]]]) * 0.35
    m = int(np.ceil(np.sqrt(n)))
    sc = scenes.Scene("side by side", iterations=1)
    sc.shapes = [scenes.cube_points(0.5), ico, scenes.box_points(m + 5.0, 1.0, m + 5.0)]
    sc.add(0.0, (0.0, -1.0, 0.0), (0.0, 0.0, 0.0, 1.0), 2)
    kind = np.zeros(n, int) if large == "none" else np.ones(n, int) if large == "all" else \
        (rng.random(n) < 0.4).astype(int)
    lift = np.where(rng.random(n) < 0.1, 0.03, -0.01)
    low = np.array([0.5, float(-ico[:, 1].min())])[kind]
    for i in range(n):
        sc.add(1.0, (2.0 * (i % m) - m, low[i] + lift[i], 2.0 * (i // m) - m),
               (0.0, 0.0, 0.0, 1.0), int(kind[i]))
    w = scenes.build_world(sc)
    s = Snapshot(w)
    w.step_partial(L.STAGE_CONSTRAINTS)
    _, _, _, pairs = oracle_broadphase(s)
    assert np.array_equal(w.pairs(), pairs)
    ref = oracle_contacts(s, pairs)
    got = w.contacts(O.CONTACT_DTYPE)
    assert len(got) == len(ref) > 0
    for f in ("pair_index", "body_a", "body_b"):
        assert np.array_equal(got[f], ref[f]), f
    assert np.array_equal(got["normal"][:, 3], ref["normal"][:, 3])
    assert w.stats()["overflow_flags"] == 0
    w.close()
