"""The mesh cull by groups of 64 triangles: meshes of 1, 63 to 65 and more than
64 x 64 triangles, in strip order and shuffled (every group then spans the
mesh), one or two of them in a world, one turned, with a compound body beside
them.  The expanded pair list equals the oracle's per-triangle test exactly."""
import numpy as np
import pytest

from experiments_amd import _lib as L
from experiments_amd import scenes
from experiments_amd.world import World, reference_config
from oracle.step import Snapshot, expand_compound_pairs, oracle_broadphase

pytestmark = pytest.mark.gpu


def strip(tris, width):
    """`tris` triangles in rows of `width` quads, 1 x 1 apart, slightly bumpy."""
    n = (tris + 1) // 2
    rows = (n + width - 1) // width
    x, z = np.meshgrid(np.arange(width + 1), np.arange(rows + 1))
    v = np.stack([x, 0.1 * np.sin(1.3 * x + 0.7 * z), z], -1).reshape(-1, 3).astype(np.float32)
    q = np.arange(n)
    a = (q // width) * (width + 1) + q % width
    t = np.stack([np.stack([a, a + width + 1, a + 1], 1),
                  np.stack([a + 1, a + width + 1, a + width + 2], 1)], 1).reshape(-1, 3)
    return v, t[:tris].astype(np.int32)


@pytest.mark.parametrize("tris", [1, 63, 64, 65, 129, 4095, 4097])
@pytest.mark.parametrize("shuffled", [False, True])
def test_expanded_pairs_match_oracle(tris, shuffled):
    rng = np.random.default_rng(tris)
    v, t = strip(tris, max(1, int(np.sqrt(tris / 2))))
    if shuffled:
        t = rng.permutation(t)
    w = World(reference_config(max_bodies=256, max_shapes=2 * tris + 64, max_pairs=1 << 15,
                               max_contacts=1 << 14, max_pairs_per_body=64))
    cube = w.add_hull(scenes.cube_points(0.5))
    m1 = w.add_concave_mesh(v, t)
    m2 = w.add_concave_mesh(v[:, [0, 1, 2]] * np.float32(0.5), t)
    pair = w.add_compound([cube, cube], [[-0.6, 0, 0], [0.6, 0, 0]], [[0, 0, 0, 1]] * 2)
    ext = v.max(0)
    w.add_body(0.0, (0, 0, 0), (0, 0, 0, 1), m1)
    for k in range(40):
        p = rng.uniform(0, 1, 3) * ext
        q = rng.normal(size=4)
        w.add_body(1.0, (p[0], rng.uniform(-0.3, 0.8), p[2]), q / np.linalg.norm(q), cube)
    w.add_body(0.0, (0.3, 0.2, -0.4), (0, np.sin(0.35), 0, np.cos(0.35)), m2)
    w.add_body(1.0, (0.5, 6.0, 0.5), (0, 0, 0, 1), pair)
    w.add_body(1.0, (0.6, 6.7, 0.7), (0, 0, 0, 1), cube)
    w.upload()
    for _ in range(2):
        s = Snapshot(w)
        w.step_partial(L.STAGE_PAIRS)
        _, _, _, pairs = oracle_broadphase(s)
        expanded = expand_compound_pairs(s, pairs)
        assert np.array_equal(w.pairs(), expanded)
        assert len(expanded) > len(pairs)
        # the turned mesh is moved: its bounds are of this step
        i = 41
        w.set_state(**{k: s.state[k] for k in ("quat", "linvel", "angvel")},
                    pos=np.where(np.arange(len(s.state["pos"]))[:, None] == i,
                                 s.state["pos"] + np.float32([0.7, 0.1, 0.3, 0]), s.state["pos"]))
    w.close()
