"""Vorticity and anisotropy over staged halos: blocks that fit the tile, blocks that do not (run table),
both in one scene, a pool, capped lists, and steps of some scenes; bit for bit against the oracle."""
import numpy as np
import pytest

import cnhip
from cnhip import scenes

from test_gpu_fluid_parity import mixed_scene, params, small_cloud
from test_gpu_vorticity import swirl

pytestmark = pytest.mark.gpu


def clumped(seed=3):
    """A thin cloud with one clump whose cells hold some 500 particles each."""
    rng = np.random.default_rng(seed)
    pts = np.concatenate([rng.random((1500, 3)) * 0.5 + 0.05, rng.random((6000, 3)) * 0.08 + 0.3])
    sc = scenes._fluid_scene(pts.astype(np.float32), 0.02, scenes.container((0, 0, 0), (0.6, 0.6, 0.6)), "clump", {})
    sc.fluid_mats = cnhip.fluid_material(0.02, vorticity_confinement=0.7)
    return swirl(sc)


def mixed():
    sc = swirl(mixed_scene())
    sc.fluid_mats = np.concatenate([cnhip.fluid_material(0.02, vorticity_confinement=0.8),
                                    cnhip.fluid_material(0.02, viscosity=50.0, vorticity_confinement=0.3)])
    return sc


def cloud(n=1500, seed=5):
    sc = swirl(small_cloud(n, seed))
    sc.fluid_mats = cnhip.fluid_material(0.02, vorticity_confinement=0.5)
    return sc


@pytest.mark.parametrize("tile", [None, 256, 700])
@pytest.mark.parametrize("build,cap", [(cloud, 64), (cloud, 5), (clumped, 40), (mixed, 64), (mixed, 7)])
def test_post_tiles_bitexact(oracle, build, cap, tile):
    sc = build()
    p = params(cap=cap, substeps=2, iters=2)
    osc = oracle.OracleScene(sc)
    want = osc.enable_render_anisotropy()
    with cnhip.Solver(0) as s:
        s.reserve(sc.n, 64)
        s.upload(sc)
        s.render_anisotropy_enable(True)
        if tile:
            s.tune_set(tile, 8)
        for k in range(2):
            print(build.__name__, cap, tile, k, flush=True)
            s.step(p)
            oracle.step(osc, p)
            np.testing.assert_array_equal(s.render_anisotropy(), want)
            pos, _, vel = s.readback()
            np.testing.assert_array_equal(pos, osc.pos)
            np.testing.assert_array_equal(vel, osc.vel)


def test_post_tiles_in_a_pool(oracle):
    solid = scenes.compose([scenes.soft_block_part(4, 0.05)], cnhip.fluid_material(0.03),
                           np.zeros(0, cnhip.COLLIDER_DTYPE), "solid")
    ses = [cloud(900, 2), solid, mixed(), cloud(1100, 4)]
    p = params(cap=64, substeps=2, iters=2)
    oscs = [oracle.OracleScene(sc) for sc in ses]
    with cnhip.Solver(0) as s:
        s.reserve(sum(sc.n for sc in ses), 64)
        s.upload_batch(ses)
        for some in (None, [2], [0, 1], None):
            s.step(p) if some is None else s.step_scenes(p, some)
            for k in range(4) if some is None else some:
                oracle.step(oscs[k], p)
            for k, o in enumerate(oscs):
                pos, _, vel = s.readback_scene(k)
                assert np.array_equal(pos, o.pos) and np.array_equal(vel, o.vel), (some, k)
