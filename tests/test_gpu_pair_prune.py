"""The narrowphase's first pass takes out pairs that are apart by more than
rounding: hull pairs from overlapping to well apart with gaps down to rounding,
near the origin and far from it, with orientations that are not quite unit.
The contacts are those of the oracle, which tests every axis."""
import numpy as np
import pytest

import oracle as O
from experiments_amd import _lib as L
from experiments_amd import scenes
from oracle.step import Snapshot, oracle_broadphase, oracle_contacts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("far", [0.0, 900.0])
@pytest.mark.parametrize("scale", [1.0, 1.0 + 4e-6, 1.002])
@pytest.mark.parametrize("verts", [4, 8, 32])
def test_contacts_equal_oracle(far, scale, verts):
    rng = np.random.default_rng(int(far) + verts)
    pts = rng.normal(size=(verts, 3))
    pts = (0.5 * pts / np.linalg.norm(pts, axis=1, keepdims=True)).astype(np.float32)
    sc = scenes.Scene("pairs", iterations=1)
    sc.shapes = [scenes.cube_points(0.5), pts]
    k = 0
    for gap in [-0.2, -1e-3, -1e-5, 0.0, 1e-7, 1e-5, 1e-4, 1e-3, 1e-2, 0.1]:
        for kind in (0, 1):
            for turn in range(4):
                at = np.array([3.0 * (k % 10) + far, far, 3.0 * (k // 10) - far])
                q = rng.normal(size=4) if turn else np.array([0.0, 0.0, 0.0, 1.0])
                q = q / np.linalg.norm(q) * scale
                # the first cube's top face, the other body above it: an
                # axis-aligned cube by its face, the rest by about a corner
                low = 0.5 if (kind == 0 and not turn) else 0.42
                sc.add(1.0, tuple(at), (0.0, 0.0, 0.0, 1.0), 0)
                sc.add(1.0, tuple(at + [0.3 * rng.random(), 0.5 + low + gap, 0.0]), tuple(q), kind)
                k += 1
    w = scenes.build_world(sc)
    s = Snapshot(w)
    w.step_partial(L.STAGE_CONSTRAINTS)
    _, _, _, pairs = oracle_broadphase(s)
    assert np.array_equal(w.pairs(), pairs)
    ref = oracle_contacts(s, pairs)
    got = w.contacts(O.CONTACT_DTYPE)
    assert 0 < len(ref) < len(pairs)
    for f in ("pair_index", "body_a", "body_b"):
        assert np.array_equal(got[f], ref[f]), f
    assert np.array_equal(got["normal"][:, 3], ref["normal"][:, 3])
    w.close()
