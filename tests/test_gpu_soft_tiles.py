"""Soft-constraint passes over tiles of particles: tile borders and remainders, particles with more
constraints than a tile holds (passes over the whole pool), degenerate tets that keep their records,
pools whose scenes run different constraint groups; bit for bit against the oracle."""
import numpy as np
import pytest

import cnhip
from cnhip import authoring as au
from cnhip import scenes

pytestmark = pytest.mark.gpu


def params(iters=3, substeps=2):
    return cnhip.default_params(dt=1 / 120, substeps=substeps, default_iterations=iters, max_fluid_neighbors=64)


def edges_of(pos, pairs, rng):
    e = np.zeros(len(pairs), au.EDGE_DTYPE)
    e["a"], e["b"] = pairs[:, 0], pairs[:, 1]
    e["rest_length"] = np.linalg.norm(pos[pairs[:, 0]] - pos[pairs[:, 1]], axis=1) * rng.uniform(0.8, 1.2, len(pairs))
    e["compliance"] = 1e-6
    e["enabled"] = rng.random(len(pairs)) > 0.05
    return e


def chain(n, seed=0):
    """n particles in random order along a line: edges, every third triple a bend, some pinned."""
    rng = np.random.default_rng(seed)
    order = rng.permutation(n)
    pos = np.zeros((n, 3), np.float32)
    pos[order] = np.stack([np.arange(n) * 0.03, rng.uniform(0.5, 0.52, n), rng.uniform(0, 0.02, n)], 1)
    part = scenes._solid_part(pos, 0.004, 20.0)
    part["pos"][rng.random(n) < 0.05, 3] = 0.0
    part["edges"] = edges_of(pos, np.stack([order[:-1], order[1:]], 1), rng)
    b = np.zeros(max(n - 2, 0) // 3, au.BEND_DTYPE)
    for k, f in enumerate(("p0", "p1", "p2")):
        b[f] = order[k:][: 3 * len(b) : 3]
    b["rest_angle"] = 2.9
    b["compliance"] = 1e-5
    part["bends"] = b
    return part


def star(leaves):
    """One heavy particle joined to all the others."""
    rng = np.random.default_rng(3)
    pos = rng.uniform(0.2, 1.4, (leaves + 1, 3)).astype(np.float32)
    part = scenes._solid_part(pos, 0.002, 20.0)
    part["pos"][0, 3] = np.float32(20.0 / leaves)
    part["edges"] = edges_of(pos, np.stack([np.zeros(leaves, int), np.arange(1, leaves + 1)], 1), rng)
    return part


def scene(*parts):
    return scenes.compose(list(parts), cnhip.fluid_material(0.03), np.zeros(0, cnhip.COLLIDER_DTYPE), "tiles")


def same(solver, oracle, sc, p, steps=3, between=None):
    osc = oracle.OracleScene(sc)
    solver.reserve(max(sc.n, 64), 64)
    solver.upload(sc)
    for k in range(steps):
        if between:
            between(k, osc)
        solver.step(p)
        oracle.step(osc, p)
        pos, _, vel = solver.readback()
        assert np.isfinite(pos).all(), k
        np.testing.assert_array_equal(pos, osc.pos, err_msg=str(k))
        np.testing.assert_array_equal(vel, osc.vel, err_msg=str(k))
    return osc


@pytest.mark.parametrize("n", [2, 3, 255, 256, 257, 513, 1500])
def test_tile_borders(solver, oracle, n):
    same(solver, oracle, scene(chain(n)), params())


@pytest.mark.parametrize("side", [362, 363])  # 131,044 and 131,769 particles: tiles of 128 and of 256
def test_tile_sizes(solver, oracle, side):
    same(solver, oracle, scene(scenes.cloth_part(side, 0.03)), params(2, 1), steps=1)


# 2,779 records with the particles at their other ends fill the LDS of a tile; past that the whole-pool passes run
@pytest.mark.parametrize("leaves", [300, 2700, 2900])
def test_star(solver, oracle, leaves):
    same(solver, oracle, scene(star(leaves), scenes.soft_block_part(4, 0.05), chain(40)), params())


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("whole_pool", [False, True])
def test_degenerate_tets_keep_their_records(oracle, graph, whole_pool):
    """Tets that solve at first and, once their compliance is set to zero, no longer (the gradients of
    a 2 cm tet stay under the threshold): their last corrections go on being applied, over substeps and
    steps, whatever their compliances become again."""
    parts = [scenes.soft_block_part(5, 0.02, mass=0.05, compliance=1e-4), chain(30)]
    if whole_pool:
        parts.append(star(3000))
    sc = scene(*parts)
    sc.tets["rest_volume"] *= np.float32(1.3)
    with cnhip.Solver(0) as solver:
        solver.graphs(graph)

        def edit(k, osc):
            if k in (2, 5):
                sc.tets["compliance"][::1 if k == 2 else 3] = np.float32(0.0 if k == 2 else 1e-4)
                solver.set_scene_constraints(0, sc)
                osc.tets[:] = sc.constraint_arrays()[3]

        osc = same(solver, oracle, sc, params(), 8, edit)
    assert np.abs(osc.vel[:, :3]).max() > 0


def test_negative_and_zero_inverse_masses(solver, oracle):
    sc = scene(scenes.soft_block_part(5, 0.05, compliance=0.0), chain(300))
    rng = np.random.default_rng(5)
    sc.pos[rng.random(sc.n) < 0.1, 3] *= np.float32(-0.5)
    sc.pos[rng.random(sc.n) < 0.1, 3] = 0.0
    same(solver, oracle, sc, params(), 2)


@pytest.mark.parametrize("iters", [1, 2, 3])
def test_pool_of_different_groups(oracle, iters):
    """Scenes with one, two and three constraint groups: each alternates its position buffers by its
    own count of groups; steps of some scenes leave the others' records and positions alone."""
    ses = [scene(star(50)), scene(chain(600)), scene(scenes.soft_block_part(7, 0.05), scenes.cloth_part(20, 0.03)),
           scene(scenes.fluid_part(4, 0.03, 0.015)), scene(scenes.cloth_part(9, 0.03))]
    p = params(iters)
    oscs = [oracle.OracleScene(s) for s in ses]
    with cnhip.Solver(0) as pool:
        pool.reserve(sum(s.n for s in ses), 64)
        pool.upload_batch(ses)
        for some in (None, [0, 2], [1], None, [4, 3, 2]):
            pool.step(p) if some is None else pool.step_scenes(p, some)
            for k in range(len(ses)) if some is None else some:
                oracle.step(oscs[k], p)
            for k, o in enumerate(oscs):
                pos, _, vel = pool.readback_scene(k)
                assert np.array_equal(pos, o.pos) and np.array_equal(vel, o.vel), (some, k)


@pytest.mark.parametrize("solves,contacts", [(1, 3), (3, 1), (2, 2)])
def test_contacts_after_the_last_group(oracle, solves, contacts):
    """Scenes whose particle-rigid contacts are solved with the tiles of their last group (edges alone,
    edges and bends, all three groups), in more and in fewer iterations than the constraints."""
    walls = scenes.container((0.05, 0.505, 0.005), (3.0, 2.0, 2.0))
    bodies = [star(300), chain(600), scenes.soft_block_part(7, 0.05, translation=(0.3, 0.7, 0.3)),
              scenes.cloth_part(20, 0.03, translation=(0.3, 0.51, 0.3)),
              scenes.soft_block_part(7, 0.05, translation=(0.25, 0.67, 0.3))]
    ses = [scenes.compose([b], cnhip.fluid_material(0.03), walls, "walls") for b in bodies]
    p = cnhip.default_params(dt=1 / 120, substeps=2, default_iterations=2, max_fluid_neighbors=64,
                             soft_internal_iterations=solves, soft_contact_iterations=contacts)
    oscs = [oracle.OracleScene(s) for s in ses]
    free = [oracle.OracleScene(scene(b)) for b in bodies]
    with cnhip.Solver(0) as pool:
        pool.reserve(sum(s.n for s in ses), 64)
        pool.upload_batch(ses)
        for some in (None, [1, 3], None):
            pool.step(p) if some is None else pool.step_scenes(p, some)
            for k in range(len(ses)) if some is None else some:
                oracle.step(oscs[k], p)
                oracle.step(free[k], p)
            for k, o in enumerate(oscs):
                pos, _, vel = pool.readback_scene(k)
                assert np.array_equal(pos, o.pos) and np.array_equal(vel, o.vel), (some, k)
    # every scene had contacts but the third, whose block hangs clear of the walls
    assert [not np.array_equal(o.pos, f.pos) for o, f in zip(oscs, free)] == [True, True, False, True, True]
