"""Fluids of few particles in many cell blocks, whose fluid passes share a CU's LDS by the blocks: sprays
around the sizes where the layout changes, alone and as a pool, with and without a viscous material, bit
for bit like the oracle."""
import numpy as np
import pytest

import cnhip
from cnhip import scenes

pytestmark = pytest.mark.gpu


def spray(n, seed, viscosity=0.01, per_cell=0.2):
    """n particles at random, per_cell to a cell (h = 0.1 m): some 64 per_cell to a block, drifting in pairs."""
    rng = np.random.default_rng(seed)
    edge = (n / per_cell * 0.1 ** 3 / 2) ** (1 / 3)
    p = rng.random((n, 3)) * np.array([2 * edge, edge, edge])
    p[1::2] = p[0::2][: n // 2] + rng.uniform(-0.04, 0.04, (n // 2, 3))  # a neighbor for every other one
    part = scenes.fluid_part(1, 0.05, 0.03)
    part = {k: np.repeat(v, n, axis=0) for k, v in part.items()}
    part["pos"][:, :3] = p
    sc = scenes.compose([part], scenes.fluid_material(0.03, viscosity=viscosity, cohesion=0.5 if viscosity > 1 else 0.0),
                        scenes.container((0.0, 0.0, 0.0), (2 * edge, edge, edge)), f"spray_{n}", {})
    sc.vel[:, :3] = rng.normal(0.0, 0.5, (n, 3)).astype(np.float32)
    return sc


def params():
    return cnhip.default_params(dt=1 / 120, substeps=2, default_iterations=4, max_fluid_neighbors=64)


@pytest.mark.parametrize("viscosity", [0.01, 40.0])
@pytest.mark.parametrize("n", [3000, 6000, 20000])  # 127, 260 and 852 blocks by the estimate
def test_spray_bitexact(solver, oracle, n, viscosity):
    sc = spray(n, n, viscosity)
    osc = oracle.OracleScene(sc)
    solver.reserve(sc.n, 64)
    solver.upload(sc)
    for s in range(2):
        print(f"{n} particles, step {s}", flush=True)
        solver.step(params())
        oracle.step(osc, params())
    pos, _, vel = solver.readback()
    np.testing.assert_array_equal(pos, osc.pos)
    np.testing.assert_array_equal(vel, osc.vel)
    assert solver.meta().max_fluid_neighbor_count > 0


def test_pool_of_sprays_and_a_block(oracle):
    scs = [spray(9000, 1), scenes.batch_scene(4000, 0, 2), spray(7000, 3), scenes.batch_scene(900, 2, 4)]
    with cnhip.Solver(0) as pool:
        pool.reserve(sum(sc.n for sc in scs), 64)
        pool.upload_batch(scs)
        for s in range(2):
            print(f"pool step {s}", flush=True)
            pool.step(params())
        got = [pool.readback_scene(k) for k in range(len(scs))]
    for k, sc in enumerate(scs):
        osc = oracle.OracleScene(sc)
        for _ in range(2):
            oracle.step(osc, params())
        np.testing.assert_array_equal(got[k][0], osc.pos, err_msg=f"scene {k}")
        np.testing.assert_array_equal(got[k][2], osc.vel, err_msg=f"scene {k}")
