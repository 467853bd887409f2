"""Pair lists into the pair array: bodies with fewer pairs than the lanes that
copy them, as many and more, beside large bodies whose lists span from none to
several workgroups, in scenes of 1 to 700 bodies, and a pair array too short for
all of them."""
import numpy as np
import pytest

from experiments_amd import _lib as L
from experiments_amd import scenes
from oracle.step import Snapshot, oracle_broadphase

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [[1], [7, 1, 9], [255, 256, 257], [1, 700, 2, 0, 40]])
@pytest.mark.parametrize("room", [1 << 15, 100])
def test_pairs_equal_oracle(counts, room):
    rng = np.random.default_rng(sum(counts))
    sc = scenes.Scene("grounds", iterations=1)
    sc.shapes = [scenes.cube_points(0.5), scenes.box_points(60.0, 1.0, 60.0)]
    for k, n in enumerate(counts):
        side = max(1.0, 1.1 * n ** (1 / 3))
        at = rng.uniform(-side / 2, side / 2, (n, 3))
        half = n // 2
        for a in at[:half]:
            sc.add(1.0, tuple(a), (0.0, 0.0, 0.0, 1.0), 0, scene=k)
        # the ground between the bodies: it lists those before it, those after list it
        sc.add(0.0, (0.0, 0.0, 0.0), (0.0, 0.0, 0.0, 1.0), 1, scene=k)
        for a in at[half:]:
            sc.add(1.0, tuple(a), (0.0, 0.0, 0.0, 1.0), 0, scene=k)
    w = scenes.build_world(sc, max_pairs_per_body=64, max_pairs=room, max_contacts=1 << 14)
    s = Snapshot(w)
    w.step_partial(L.STAGE_PAIRS)
    pairs = oracle_broadphase(s)[3]
    assert np.array_equal(w.pairs(), pairs[:room])
    over = bool(w.stats()["overflow_flags"] & L.OVERFLOW_PAIRS)
    assert over == (len(pairs) > room)
    w.close()
