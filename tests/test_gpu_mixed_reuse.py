"""Candidate lists in scenes whose contacts move fluid particles too: a tet block pressed and shot into
fluid, so that contact corrections stay inside the lists' allowance or exceed it, over more and fewer
contact than fluid iterations; bit for bit against the oracle."""
import numpy as np
import pytest

import cnhip
from cnhip import scenes

pytestmark = pytest.mark.gpu


def pressed(speed):
    block = scenes.soft_block_part(6, 0.04, translation=(0.3, 0.3, 0.3))
    cloth = scenes.cloth_part(10, 0.03, translation=(0.1, 0.2, 0.1))
    fluid = scenes.fluid_part(15, 0.03, 0.018, seed=4, jitter=0.005)
    sc = scenes.compose([block, cloth, fluid], cnhip.fluid_material(0.018),
                        scenes.container((0, 0, 0), (0.6, 0.8, 0.6)), "pressed")
    sc.vel[: len(block["pos"]), 1] = -speed
    return sc


def run(solver, oracle, sc, contacts, steps=3):
    p = cnhip.default_params(dt=1 / 120, substeps=4, default_iterations=4, max_fluid_neighbors=64,
                             soft_contact_iterations=contacts)
    osc = oracle.OracleScene(sc)
    solver.reserve(sc.n, 64)
    solver.upload(sc)
    reuses = 0
    for _ in range(steps):
        solver.step(p)
        oracle.step(osc, p)
        reuses += solver.meta().candidate_reuses
        pos, _, vel = solver.readback()
        assert np.isfinite(pos).all()
        np.testing.assert_array_equal(pos, osc.pos)
        np.testing.assert_array_equal(vel, osc.vel)
    most = steps * 4 * 3 * int((sc.kinds == cnhip.CN_PARTICLE_KIND_FLUID).sum())
    print(sc.name, "contacts", contacts, "reuses", reuses, "of", most, flush=True)
    return reuses, most


@pytest.mark.parametrize("contacts", [1, 3, 6])
@pytest.mark.parametrize("speed", [0.0, 2.0, 40.0])
def test_lists_follow_contacts(solver, oracle, speed, contacts):
    reuses, most = run(solver, oracle, pressed(speed), contacts)
    assert reuses < most  # some blocks moved too far


@pytest.mark.parametrize("contacts", [0, 2, 6])
def test_calm_scene_reuses_its_lists(solver, oracle, contacts):
    reuses, _ = run(solver, oracle, scenes.mixed(14, 6, 20), contacts)
    assert reuses > 0
