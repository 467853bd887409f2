"""Batched scenes at the edges of the solver's size classes: scenes of 1 to
1,100 rows alone on a compute unit (two or three rows held per four lanes, or
read on every pass; more bodies than the velocity cache holds), and 4,096
scenes, where small ones share a workgroup.  One step equals the oracle's
per-scene solve on the GPU's constraint order; the operations are the same
one by one, so the tolerance is a few roundings of the velocities."""
import numpy as np
import pytest

import oracle as O
from experiments_amd import _lib as L
from experiments_amd import scenes
from oracle.step import Snapshot, gpu_tile_orders, oracle_step

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

EDGES = [1, 31, 33, 64, 65, 128, 129, 256, 257, 512, 513, 768, 769, 1100]
SMALL = [1, 2, 15, 16, 17, 31, 32, 33, 1, 1, 2, 3]


def columns(counts):
    """One scene per count: that many cubes resting in columns on its ground,
    one contact per cube."""
    sc = scenes.Scene("columns", iterations=3)
    sc.shapes = [scenes.cube_points(0.5), scenes.box_points(12.0, 1.0, 12.0)]
    rng = np.random.default_rng(5)
    for s, n in enumerate(counts):
        sc.add(0.0, (0.0, -1.0, 0.0), (0.0, 0.0, 0.0, 1.0), 1, s)
        m = int(np.ceil(n ** (1 / 3.0)))
        for b in range(n):
            j, c = divmod(b, m * m)
            x, z = (c % m - (m - 1) / 2) * 1.05, (c // m - (m - 1) / 2) * 1.05
            sc.add(1.0, (x, 0.495 + 0.993 * j, z), (0.0, 0.0, 0.0, 1.0), 0, s,
                   tuple(0.2 * rng.normal(size=3)))
    return sc


@pytest.mark.parametrize("layout", ["edges", "shared"])
@pytest.mark.parametrize("block", [256, 512])
@pytest.mark.parametrize("tol", [0.0, 1e-2])
def test_step_matches_oracle(layout, block, tol):
    counts = EDGES if layout == "edges" else (EDGES[4:9] * 2 + SMALL * 400)[:4096]
    if layout == "shared":
        counts += [1] * (4096 - len(counts))
    w = scenes.build_world(columns(counts), max_pairs_per_body=64, residual_tolerance=tol,
                           solver_iterations=3 if tol == 0.0 else 20)
    w.set_tuning(solve_block=block)
    s = Snapshot(w)
    w.step_partial(L.STAGE_COLOR)
    segs = gpu_tile_orders(w)
    rows = sorted({len(x) for x in segs})
    assert rows == sorted(set(counts)), rows
    contacts = w.contacts(O.CONTACT_DTYPE)
    w.set_state(**{k: s.state[k] for k in ("pos", "quat", "linvel", "angvel")})
    w.step(1)
    assert w.stats()["overflow_flags"] == 0
    g = w.get_state()
    ref = oracle_step(s, None, contacts, segments=segs)
    for k in ("linvel", "angvel"):
        assert np.allclose(g[k][:, :3], ref[k][:, :3], rtol=2e-6, atol=2e-6), k
    if tol > 0.0:
        st = w.read(L.BUF_TILE_STATS, np.int32, (4,))
        assert np.array_equal(st[:, :2], np.array(ref["iters"]).reshape(-1, 2))
    w.close()


def test_batched_worlds_hold_no_packed_rows():
    """Only spatial tiles read packed rows (41 float4 a contact): a batched
    world with the same room holds less device memory by them."""
    room, held = 1 << 20, []
    for scene in (0, 1):
        sc = columns([8])
        sc.add(0.0, (40.0, -1.0, 0.0), (0.0, 0.0, 0.0, 1.0), 1, scene)
        free = torch.cuda.mem_get_info()[0]
        w = scenes.build_world(sc, max_contacts=room)
        held.append(free - torch.cuda.mem_get_info()[0])
        w.step(1)
        assert w.stats()["num_contacts"] == 8
        w.close()
    assert held[0] - held[1] >= 0.95 * 41 * 16 * room


@pytest.mark.parametrize("n_scenes", [1, 8])
def test_autotune_times_a_shape_once(n_scenes):
    """Where no scenes share a workgroup solve_block changes nothing: it stays,
    and its two halves of the candidates are the same measurements."""
    w = scenes.build_world(columns([8] * n_scenes))
    w.set_tuning(solve_block=512)
    best, ms = w.autotune(steps=2)
    assert best["solve_block"] == 512 and w.get_tuning()["solve_block"] == 512
    for waves in (2, 4, 6, 8):
        assert ms["256/%d" % waves] == ms["512/%d" % waves] > 0.0
    w.close()
