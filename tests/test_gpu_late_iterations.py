"""Pools past the 64 iterations whose fluid passes run over cell blocks: from there on a thread takes a
slot and a wave at a scenes' border holds particles of two, each of which has its own scene's colliders.
Scenes of odd counts with different walls step bit for bit like the oracle."""
import numpy as np
import pytest

import cnhip
from cnhip import scenes

pytestmark = pytest.mark.gpu


def room(side, box, seed, pegs=False):
    """A fluid block filling the corner of its own container; with pegs: more than 32 colliders."""
    part = scenes.fluid_part(side, 0.05, 0.03, origin=(0.0, 0.0, 0.0), seed=seed, jitter=0.005)
    sc = scenes.compose([part], scenes.fluid_material(0.03), scenes.container((0.0, 0.0, 0.0), box),
                        f"room_{side}_{seed}", {})
    if pegs:
        sc.shape_colliders = scenes.pegboard_colliders(7, 5, y=0.15, spacing=0.1, origin=(0.05, 0.05))
    return sc


def batch():
    return [room(7, (0.36, 1.0, 0.5), 1), room(9, (0.46, 0.8, 0.44), 2, pegs=True), room(5, (0.3, 0.5, 0.26), 3),
            room(8, (2.0, 0.7, 0.41), 4)]


@pytest.mark.parametrize("iterations", [64, 66])
@pytest.mark.parametrize("ids", [None, [0, 2, 3]])
def test_pool_at_many_iterations(oracle, iterations, ids):
    scs = batch()
    assert all(sc.n % 64 for sc in scs[:3])
    p = cnhip.default_params(dt=1 / 120, substeps=1, default_iterations=iterations, max_fluid_neighbors=64)
    steps = 2
    with cnhip.Solver(0) as pool:
        pool.reserve(sum(sc.n for sc in scs), 64)
        pool.upload_batch(scs)
        for s in range(steps):
            print(f"step {s} of {iterations} iterations, scenes {ids}", flush=True)
            if ids is None:
                pool.step(p)
            else:
                pool.step_scenes(p, ids)
        got = [pool.readback_scene(k) for k in range(len(scs))]
    for k, sc in enumerate(scs):
        osc = oracle.OracleScene(sc)
        for _ in range(steps if ids is None or k in ids else 0):
            oracle.step(osc, p)
        np.testing.assert_array_equal(got[k][0], osc.pos, err_msg=f"scene {k}")
        np.testing.assert_array_equal(got[k][2], osc.vel, err_msg=f"scene {k}")
