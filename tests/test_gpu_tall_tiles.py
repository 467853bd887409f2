"""Spatial solver tiles of tall columns, at the row counts where a tile's rows
fit the quads of its 256 threads (up to 128 bodies) or 512 threads (more) once,
twice or not at all: one step equals the oracle's on the GPU's constraint order.
The operations are the same one by one, so the tolerance is a few roundings of
the velocities."""
import numpy as np
import pytest

import oracle as O
from experiments_amd import _lib as L
from experiments_amd import scenes
from oracle.step import Snapshot, gpu_order, oracle_step

pytestmark = pytest.mark.gpu


def columns(height, iters):
    """Four columns of cubes in one solver tile, one contact per cube."""
    sc = scenes.Scene("columns", iterations=iters)
    sc.shapes = [scenes.cube_points(0.5), scenes.box_points(12.0, 1.0, 12.0)]
    rng = np.random.default_rng(height)
    sc.add(0.0, (0.0, -1.0, 0.0), (0.0, 0.0, 0.0, 1.0), 1)
    for j in range(height):
        for c in range(4):
            sc.add(1.0, (1.05 * (c % 2), 0.495 + 0.993 * j, 1.05 * (c // 2)), (0.0, 0.0, 0.0, 1.0), 0,
                   0, tuple(0.2 * rng.normal(size=3)))
    return sc


@pytest.mark.parametrize("height,tol", [(h, 0.0) for h in (1, 16, 17, 32, 33, 64, 65, 128, 129, 260)] +
                         [(h, 1e-2) for h in (33, 65)])
def test_step_matches_oracle(height, tol):
    w = scenes.build_world(columns(height, 3), tile_size=4.0, max_pairs_per_body=64,
                           residual_tolerance=tol)
    s = Snapshot(w)
    w.step_partial(L.STAGE_COLOR)
    order = gpu_order(w)
    contacts = w.contacts(O.CONTACT_DTYPE)
    assert len(contacts) == 4 * height
    w.set_state(**{k: s.state[k] for k in ("pos", "quat", "linvel", "angvel")})
    w.step(1)
    assert w.stats()["overflow_flags"] == 0
    g = w.get_state()
    ref = oracle_step(s, order, contacts)
    for k in ("linvel", "angvel"):
        assert np.allclose(g[k][:, :3], ref[k][:, :3], rtol=2e-6, atol=2e-6), k
    w.close()
