"""Neighbor lists held four entries to a word: caps that cut a word, lists that overflow the cap or the
candidate slots, every combination of delta terms and layouts, and a viscosity edit under a captured
graph, bit for bit against the oracle."""
import numpy as np
import pytest

import cnhip
from cnhip import scenes

pytestmark = pytest.mark.gpu


def squeezed(side, factor, seed=0, **material):
    """A dam-break lattice pressed together by `factor` (more neighbors, larger halos)."""
    sc = scenes.dam_break_64k(seed=seed, side=side)
    sc.pos[:, :3] *= np.float32(factor)
    sc.fluid_mats = cnhip.fluid_material(0.03, **material)
    return sc


def check(solver, oracle, sc, p, steps=2):
    osc = oracle.OracleScene(sc)
    solver.reserve(sc.n, max(64, p.max_fluid_neighbors))
    solver.upload(sc)
    for _ in range(steps):
        solver.step(p)
        st = oracle.step(osc, p)
        m = solver.meta()
        assert m.fluid_neighbor_truncations == st.truncations
    pos, _, vel = solver.readback()
    assert np.isfinite(pos).all()
    np.testing.assert_array_equal(pos, osc.pos)
    np.testing.assert_array_equal(vel, osc.vel)


@pytest.mark.parametrize("cap", [1, 3, 4, 29, 66, 130])
@pytest.mark.parametrize("factor", [1.0, 0.7])
def test_list_caps(solver, oracle, cap, factor):
    """factor 0.7: some 80 neighbors, so most caps truncate and candidate lists (96) overflow."""
    p = cnhip.default_params(dt=1 / 480, substeps=2, default_iterations=3, max_fluid_neighbors=cap)
    print("cap", cap, "factor", factor, flush=True)
    check(solver, oracle, squeezed(9, factor), p)


TERMS = [dict(), dict(viscosity=50.0), dict(cohesion=0.5), dict(surface_tension=5000.0),
         dict(viscosity=50.0, cohesion=0.5, surface_tension=5000.0), dict(cfl_coefficient=0.01)]


@pytest.mark.parametrize("terms", TERMS, ids=lambda t: "-".join(t) or "plain")
@pytest.mark.parametrize("tile", [256, 1200, 4096])
def test_delta_terms_and_layouts(solver, oracle, terms, tile):
    """tile 1200: between the halos of a lattice's blocks; 256: every inner block walks."""
    p = cnhip.default_params(dt=1 / 240, substeps=2, default_iterations=3, max_fluid_neighbors=64)
    print(terms, tile, flush=True)
    solver.tune_set(tile, 16)
    try:
        check(solver, oracle, squeezed(11, 0.95, **terms), p)
    finally:
        solver.tune_set(4096, 1024)


def test_viscosity_edit_under_a_graph(oracle):
    """The delta pass's layout follows the largest viscosity: an edit drops the captured graph."""
    p = cnhip.default_params(dt=1 / 240, substeps=2, default_iterations=3, max_fluid_neighbors=64)
    sc = squeezed(10, 0.95)
    with cnhip.Solver(0) as s:
        s.reserve(sc.n, 64)
        s.upload(sc)
        s.graphs(True)
        osc = oracle.OracleScene(sc)
        for visc in (0.01, 50.0, 0.01):
            fm = cnhip.fluid_material(0.03, viscosity=visc)
            s.set_scene_materials(0, fluid_mats=fm)
            osc.fluid_mats[:] = fm
            for _ in range(3):
                s.step(p)
                oracle.step(osc, p)
        pos, _, vel = s.readback()
    np.testing.assert_array_equal(pos, osc.pos)
    np.testing.assert_array_equal(vel, osc.vel)
