"""Contact partners taken cell block by cell block: blocks in which no pair can exist, blocks past the
stored halo descriptors, blocks of wrapped Morton cells and hash keys, bit for bit against the oracle."""
import numpy as np
import pytest

import cnhip
from cnhip import scenes

pytestmark = pytest.mark.gpu


def clusters(centers, seed, groups=2, self_collide=False):
    """At every centre a few overlapping free solid particles of `groups` phase groups and one fluid
    particle (r = 0.01 m, cell 0.0333 m); every third centre holds one group only (no pair)."""
    rng = np.random.default_rng(seed)
    parts = []
    for g in range(groups):
        keep = centers if g == 0 else centers[np.arange(len(centers)) % 3 != 0]
        p = (keep + rng.uniform(-0.006, 0.006, keep.shape)).astype(np.float32)
        part = scenes._solid_part(np.concatenate([p, p + np.float32(0.004)]), 0.01, 1.0)
        part["self_collide"] = self_collide
        parts.append(part)
    fl = scenes.fluid_part(1, 0.02, 0.01)
    keep = centers[np.arange(len(centers)) % 3 == 1]
    n = len(keep)
    fluid = {k: np.repeat(v, n, axis=0) for k, v in fl.items()}
    fluid["pos"][:, :3] = keep + rng.uniform(-0.006, 0.006, keep.shape)
    return scenes.compose(parts + [fluid], cnhip.fluid_material(0.01), np.zeros(0, cnhip.COLLIDER_DTYPE), "clusters")


def grid(nx, ny, nz, step):
    return np.stack(np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz), indexing="ij"), -1).reshape(-1, 3) * step


CASES = {
    # a lattice finer than the blocks: pairs across block borders, blocks with and without pairs
    "dense": (lambda: grid(14, 5, 9, 0.021), {}),
    # one cluster per block and more blocks than descriptors (max(256, particles / 32))
    "sparse": (lambda: grid(9, 7, 7, 0.2), {}),
    # clusters 1,024 cells apart share Morton codes: their runs are filtered by cell
    "wrapped": (lambda: np.concatenate([grid(6, 3, 3, 0.021), grid(6, 3, 3, 0.021) + [34.133, 0.0, 0.0]]), {}),
    "self": (lambda: grid(6, 5, 4, 0.021), dict(groups=1, self_collide=True)),
    "hash": (lambda: grid(6, 5, 4, 0.021), {}),
}


@pytest.mark.parametrize("name", list(CASES))
def test_contact_blocks_bitexact(solver, oracle, name):
    centers, kw = CASES[name]
    sc = clusters(centers(), 5, **kw)
    p = cnhip.default_params(dt=1 / 120, substeps=2, default_iterations=3, max_fluid_neighbors=64,
                             key_mode=cnhip.CN_KEY_HASH if name == "hash" else cnhip.CN_KEY_MORTON)
    print(name, sc.n, "particles", flush=True)
    with cnhip.Solver(0) as s:  # reserved to the scene's size: its descriptors are max(256, n / 32)
        s.reserve(sc.n, 64)
        s.upload(sc)
        osc = oracle.OracleScene(sc)
        start = sc.pos.copy()
        for _ in range(2):
            s.step(p)
            st = oracle.step(osc, p)
            assert s.meta().contact_overflows == st.contact_overflows
        pos, _, vel = s.readback()
    assert np.isfinite(pos).all() and (pos[:, 0] != start[:, 0]).any()  # contacts act along x too
    np.testing.assert_array_equal(pos, osc.pos)
    np.testing.assert_array_equal(vel, osc.vel)
