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


def at_edge(k):
    """Cubes turned 45 degrees about z, the second one k / 64 further on x and
    on y: face to face with a gap of sqrt(2) k / 64 - 1 and overlapping boxes."""
    return [(0.0, 0.0, 0.0), (k / 64.0, k / 64.0, 0.0)], np.sqrt(2.0) * k / 64.0 - 1.0


@pytest.mark.parametrize("far", [0.0, 10000.0, 100000.0])
def test_far_pairs_are_taken_out(far):
    """A pair that is apart by more than the rounding of the projections, 4
    roundings of each position's length and 1e-4 of the bodies' sizes and
    distance, does not reach the next pass, at the origin and far from it
    (positions are multiples of 1/64, so the pairs are the same ones)."""
    sc = scenes.Scene("edges", iterations=1)
    sc.shapes = [scenes.cube_points(0.5)]
    q = (0.0, 0.0, float(np.sin(np.pi / 8)), float(np.cos(np.pi / 8)))
    left = 0
    gaps = range(40, 90)
    for i, k in enumerate(gaps):
        pos, gap = at_edge(k)
        at = np.array([4.0 * (i % 10) + far, 4.0 * (i // 10) + far, far])
        for p in pos:
            sc.add(1.0, tuple(at + p), q, 0)
        lim = 2 * np.linalg.norm(at) * 4 * 2.0 ** -24 + 1e-4 * (2 * k / 64.0 + 2 * 1.5)
        left += gap <= 1.1 * lim
    w = scenes.build_world(sc)
    w.step_partial(L.STAGE_CONSTRAINTS)
    st = w.stats()
    assert st["num_pairs"] == len(gaps)
    assert st["face_pass_pairs"] <= left
    w.close()


@pytest.mark.parametrize("far", [10000.0, 100000.0])
@pytest.mark.parametrize("verts", [8, 32])
def test_far_contacts_equal_oracle(far, verts):
    """Hulls in random poses around touching: pass 0 takes out no pair that
    every axis of the oracle's test leaves overlapping."""
    rng = np.random.default_rng(int(far) + verts)
    pts = rng.normal(size=(verts, 3))
    pts = (0.5 * pts / np.linalg.norm(pts, axis=1, keepdims=True)).astype(np.float32)
    sc = scenes.Scene("far", iterations=1)
    sc.shapes = [scenes.cube_points(0.5), pts]
    for k in range(500):
        at = np.array([3.0 * (k % 25) + far, far, 3.0 * (k // 25) - far])
        d = rng.normal(size=3)
        d *= rng.uniform(0.7, 1.2) / np.linalg.norm(d)
        for p, shape in ((at, k % 2), (at + d, 1)):
            q = rng.normal(size=4)
            sc.add(1.0, tuple(p), tuple(q / np.linalg.norm(q)), shape)
    w = scenes.build_world(sc)
    s = Snapshot(w)
    w.step_partial(L.STAGE_CONSTRAINTS)
    _, _, _, pairs = oracle_broadphase(s)
    assert np.array_equal(w.pairs(), pairs)
    ref = oracle_contacts(s, pairs)
    got = w.contacts(O.CONTACT_DTYPE)
    assert 50 < len(ref) < len(pairs) - 50
    for f in ("pair_index", "body_a", "body_b"):
        assert np.array_equal(got[f], ref[f]), f
    assert np.array_equal(got["normal"][:, 3], ref["normal"][:, 3])
    w.close()
