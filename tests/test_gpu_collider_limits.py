"""Scenes at the border between candidate masks and candidate lists (31, 32 and 33 static colliders, every
one of them in reach): fluid and cloth step bit for bit like the oracle, alone and in a pool."""
import numpy as np
import pytest

import cnhip
from cnhip import scenes

pytestmark = pytest.mark.gpu


def params(**kw):
    return cnhip.default_params(dt=1 / 120, substeps=2, default_iterations=3, max_fluid_neighbors=64, **kw)


def studded(colliders, seed=0):
    """Fluid filling a floor corner around small pegs, and a cloth lying on them; with the walls that many
    colliders."""
    fluid = scenes.fluid_part(9, 0.05, 0.03, origin=(0.0, 0.0, 0.0), seed=seed, jitter=0.005)
    cloth = scenes.cloth_part(10, 0.05, 0.02, translation=(0.0, 0.12, 0.5))
    sc = scenes.compose([cloth, fluid], scenes.fluid_material(0.03), scenes.container((0.0, 0.0, 0.0), (0.47, 0.5, 1.0)),
                        f"studded_{colliders}", {})
    pegs = scenes.pegboard_colliders(6, 5, y=0.1, spacing=0.08, origin=(0.03, 0.03))
    sc.shape_colliders = pegs[:colliders - len(sc.colliders)]
    return sc


@pytest.mark.parametrize("colliders", [31, 32, 33])
def test_scene_alone(solver, oracle, colliders):
    sc = studded(colliders)
    assert len(sc.colliders) + len(sc.shape_colliders) == colliders
    osc = oracle.OracleScene(sc)
    solver.reserve(sc.n, 64)
    solver.upload(sc)
    for s in range(4):
        print(f"{colliders} colliders, step {s}", flush=True)
        solver.step(params())
        oracle.step(osc, params())
    pos, _, vel = solver.readback()
    np.testing.assert_array_equal(pos, osc.pos)
    np.testing.assert_array_equal(vel, osc.vel)
    # every peg is within the smoothing radius (0.1 m) of some fluid particle
    fluid = osc.pos[sc.kinds == 1, :3]
    for col in sc.shape_colliders:
        assert min(oracle.collider_contact(col, q)[1] for q in fluid) < 0.1


def test_pool_of_both_kinds(oracle):
    scs = [studded(32, 1), studded(31, 2), scenes.batch_scene(700, 0, 3), studded(33, 4)]
    with cnhip.Solver(0) as pool:
        pool.reserve(sum(sc.n for sc in scs), 64)
        pool.upload_batch(scs)
        for s in range(3):
            print(f"pool step {s}", flush=True)
            pool.step(params())
        got = [pool.readback_scene(k) for k in range(len(scs))]
    for k, sc in enumerate(scs):
        osc = oracle.OracleScene(sc)
        for _ in range(3):
            oracle.step(osc, params())
        np.testing.assert_array_equal(got[k][0], osc.pos, err_msg=f"scene {k}")
        np.testing.assert_array_equal(got[k][2], osc.vel, err_msg=f"scene {k}")


@pytest.mark.parametrize("colliders", [31, 32, 33])
def test_edits_across_the_border(solver, oracle, colliders):
    """Walls switched off, moved and back on: the enabled colliders of a scene cross the border both ways."""
    sc = studded(colliders, 5)
    osc = oracle.OracleScene(sc)
    solver.reserve(sc.n, 64)
    solver.upload(sc)
    for s, (off, dx) in enumerate([(0, 0.0), (2, 0.0), (1, 0.03), (0, 0.03)]):
        print(f"{colliders} colliders, {off} off", flush=True)
        cols = sc.colliders.copy()
        cols["center"][0] += np.float32(dx)
        cols["enabled"][len(cols) - off:] = 0
        solver.set_scene_colliders(0, cols)
        osc.colliders[:] = cols
        solver.step(params())
        oracle.step(osc, params())
        pos, _, vel = solver.readback()
        np.testing.assert_array_equal(pos, osc.pos, err_msg=f"edit {s}")
        np.testing.assert_array_equal(vel, osc.vel, err_msg=f"edit {s}")
