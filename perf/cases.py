"""The workloads whose speed this repository answers for, through the calls a user's program makes.

Each case is one resident scene (or pool of scenes) stepped on the GPU: a simulation that is stepped
from a known state, an environment that is reset from tensors and stepped, a served pool of which a
few sessions are stepped, and the pair sort that callers run on their own device arrays.  ``prepare``
builds and uploads the scene and keeps the solver; ``run`` is one frame: the reset, ``step`` (or
``step_scenes``) and the zero-copy views of the resulting particle state.
"""
from __future__ import annotations

import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cressim-neo_amd"))

import cnhip  # noqa: E402
from cnhip import scenes  # noqa: E402

#: particles the exact 64-bit step handles in reasonable time
EXACT_MOST = 70_000


def _case(name, kind, n, *, substeps=4, iterations=4, cap=64, graph=False, warm=0, **more):
    return dict(name=name, kind=kind, n=n, substeps=substeps, iterations=iterations, cap=cap, graph=graph, warm=warm, **more)


def listed():
    return [
        # a small interactive scene with the solver's default parameters (one substep, 20 iterations,
        # 128 neighbor slots): a frame of few particles, where launches and latency count
        _case("fluid_1728", "lattice", 12, substeps=1, iterations=20, cap=128),
        # the 64,000-particle dam break, its step captured once and replayed
        _case("fluid_64k", "lattice", 40, graph=True),
        # a viscous liquid with cohesion and surface tension, an odd particle count
        _case("viscous_300k", "fill", 300_007, warm=4, radius=0.03, viscosity=50.0, cohesion=0.5, tension=5000.0),
        # the large random fill at rest density, a few steps in
        _case("fluid_4m", "fill", 4_194_304, warm=4),
        # the same fluid after it has slumped: more neighbors, unequal cell blocks
        _case("fluid_settled_1m", "fill", 1_048_573, warm=36),
        # a rendered fluid: vorticity confinement and the anisotropy frames the renderer reads back
        _case("render_200k", "fill", 200_003, warm=4, radius=0.03, vorticity=0.6, anisotropy=True),
        # fluid, tet soft body and cloth in one scene, with contacts between them
        _case("mixed_360k", "mixed", 64, graph=True, warm=4, tet=32, cloth=256),
        # one cloth, and one tet soft body (the solids of the batched workload, alone)
        _case("cloth_64k", "cloth", 64_009, graph=True),
        _case("soft_33k", "tet", 32_768, graph=True),
        # a vectorized environment: a pool of independent scenes stepped together, episodes ending
        # in turn
        _case("pool_48", "pool", 48, graph=True, warm=2, lo=2000, hi=64000, resets=3, layout=3),
        # serving: each tick steps the few sessions that asked for a step, one of them starting anew
        _case("serve_4_of_32", "serve", 32, warm=1, lo=2000, hi=32000, tick=4, resets=1, layout=5),
        # a caller's own (key, index) pairs, sorted in place without allocation
        _case("sort_1m", "sort", 1_000_003),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["lattice", "fill", "fill", "liquid", "render", "mixed", "cloth", "tet", "pool", "serve", "sort"])
    substeps, iterations, cap = rng.choice([(4, 4, 64), (4, 4, 64), (2, 6, 64), (1, 20, 128)])
    p = dict(substeps=substeps, iterations=iterations, cap=cap, graph=rng.random() < 0.5)
    if kind == "lattice":
        c = _case("", "lattice", rng.randint(8, 40), **p)
    elif kind == "fill":
        p.update(substeps=4, iterations=4, cap=64)
        c = _case("", "fill", _log_uniform(rng, 20_000, 2_500_000) | 1, warm=rng.choice([4, 12]), **p)
    elif kind == "liquid":
        p.update(substeps=4, iterations=4, cap=64)
        c = _case("", "fill", _log_uniform(rng, 20_000, 500_000), warm=4, radius=rng.choice([0.02, 0.03]),
                  viscosity=rng.choice([0.01, 20.0, 50.0]), cohesion=rng.choice([0.0, 0.5]),
                  tension=rng.choice([0.0, 5000.0]), **p)
    elif kind == "render":
        p.update(substeps=4, iterations=4, cap=64)
        c = _case("", "fill", _log_uniform(rng, 20_000, 300_000), warm=4, radius=rng.choice([0.02, 0.03]),
                  vorticity=rng.choice([0.0, 0.6]), anisotropy=True, **p)
    elif kind == "mixed":
        p.update(substeps=4, iterations=4, cap=64)
        c = _case("", "mixed", rng.randint(16, 56), warm=4, tet=rng.randint(6, 28), cloth=rng.randint(24, 220), **p)
    elif kind in ("cloth", "tet"):
        c = _case("", kind, _log_uniform(rng, 2000, 64_000), **p)
    elif kind == "pool":
        p.update(substeps=4, iterations=4, cap=64)
        c = _case("", "pool", rng.randint(8, 48), warm=2, lo=2000, hi=rng.choice([16_000, 64_000]),
                  resets=rng.randint(1, 3), layout=rng.randrange(1000), **p)
    elif kind == "serve":
        p.update(substeps=4, iterations=4, cap=64, graph=False)
        c = _case("", "serve", rng.randint(12, 32), warm=1, lo=2000, hi=rng.choice([8000, 32_000]),
                  tick=rng.randint(1, 6), resets=1, layout=rng.randrange(1000), **p)
    else:
        c = _case("", "sort", _log_uniform(rng, 1000, 1 << 20))
    del c["name"]
    return c


def _scene(case, seed):
    kind, n = case["kind"], case["n"]
    if kind == "lattice":
        return scenes.dam_break_64k(seed=seed, side=n)
    if kind == "fill":
        box = scenes.scaled_box_for(n)
        if "radius" in case:  # the same fill of larger particles (and a box as much larger)
            scale = case["radius"] / scenes.random_fill_radius(n, float(np.prod(box)))
            box = tuple(scale * b for b in box)
        sc = scenes.large_pbf(n, seed=seed, box=box)
        sc.fluid_mats = cnhip.fluid_material(
            float(sc.radii[0]), viscosity=case.get("viscosity", 0.01), cohesion=case.get("cohesion", 0.0),
            surface_tension=case.get("tension", 0.0), vorticity_confinement=case.get("vorticity", 0.0))
        return sc
    if kind == "mixed":
        return scenes.mixed(n, case["tet"], case["cloth"], seed=seed)
    sc = scenes.batch_scene(n, {"tet": 1, "cloth": 2}[kind], seed)
    # a body in motion: its vertices off their rest places by a few percent of the spacing
    g = np.random.Generator(np.random.PCG64(seed))
    sc.pos[:, :3] += g.uniform(-0.05, 0.05, (sc.n, 3)).astype(np.float32) * (2.0 * sc.radii[:, None])
    sc.vel[:, :3] = g.normal(0.0, 0.1, (sc.n, 3)).astype(np.float32)
    return sc


def _params(case):
    return cnhip.default_params(dt=1 / 120, substeps=case["substeps"], default_iterations=case["iterations"],
                                max_fluid_neighbors=case["cap"])


def prepare(case, seed):
    if case["kind"] == "sort":
        g = torch.Generator(device="cuda").manual_seed(seed)
        keys = torch.randint(-2**31, 2**31, (case["n"],), generator=g, device="cuda", dtype=torch.int64).to(torch.int32)
        idx = torch.randperm(case["n"], generator=g, device="cuda").to(torch.int32)
        solver = cnhip.Solver(0)
        return dict(kind="sort", solver=solver, n=case["n"], keys=keys, idx=idx, k=keys.clone(), v=idx.clone(), stream=None)
    solver = cnhip.Solver(0)
    st = dict(kind=case["kind"], solver=solver, params=_params(case), frame=0, aniso=bool(case.get("anisotropy")))
    if case["kind"] in ("pool", "serve"):
        sizes, kinds = scenes.batch_sizes(case["n"], case["layout"], case["lo"], case["hi"])
        world = [scenes.batch_scene(int(m), int(k), seed + j) for j, (m, k) in enumerate(zip(sizes, kinds))]
        solver.reserve(sum(s.n for s in world), case["cap"])
        solver.upload_batch(world)
        g = np.random.Generator(np.random.PCG64(seed))
        home = []
        for s in world:
            s.vel[:, :3] = g.normal(0.0, 0.1, (s.n, 3)).astype(np.float32)
            home.append((torch.from_numpy(s.pos).cuda(), torch.from_numpy(s.vel).cuda()))
        st.update(home=home, resets=case["resets"], tick=case.get("tick", 0))
        for k, (p, v) in enumerate(home):
            solver.set_scene_state(k, p, v)
    else:
        sc = _scene(case, seed)
        solver.reserve(sc.n, case["cap"])
        solver.upload(sc)
    solver.graphs(case["graph"])
    if st["aniso"]:
        solver.render_anisotropy_enable()
    st["stream"] = solver.torch_stream()
    for _ in range(case["warm"]):
        solver.step(st["params"])
    solver.synchronize()
    st["views"] = solver.torch_views()
    if "home" not in st:
        st["home"] = [(st["views"]["positions_inv_mass"].clone(), st["views"]["velocities"].clone())]
    return st


def run(state):
    solver, stream = state["solver"], state["stream"]
    now = torch.cuda.current_stream()
    if state["kind"] == "sort":
        state["k"].copy_(state["keys"])
        state["v"].copy_(state["idx"])
        # the sort runs on the context's stream: this one waits for the copies
        now.synchronize()
        solver.pass_sort_device_noalloc(state["k"].data_ptr(), state["v"].data_ptr(), state["n"])
        solver.synchronize()
        return state["k"], state["v"]
    frame, home = state["frame"], state["home"]
    state["frame"] = frame + 1
    if state["kind"] == "serve":
        asked = [(frame * state["tick"] + j) % len(home) for j in range(state["tick"])]
        k = asked[frame % len(asked)]
        solver.set_scene_state(k, *home[k])
        solver.step_scenes(state["params"], sorted(set(asked)))
    elif state["kind"] == "pool":
        for j in range(state["resets"]):
            k = (frame * state["resets"] + j) % len(home)
            solver.set_scene_state(k, *home[k])
        solver.step(state["params"])
    else:
        solver.set_scene_state(0, *home[0])
        solver.step(state["params"])
    now.wait_stream(stream)
    out = dict(state["views"])
    if state["aniso"]:
        out["anisotropy"] = solver.render_anisotropy()
    return out


def _counts(case):
    """Particles that a pass steps (fluid, solid) and their constraints (edges, dihedrals, tets)."""
    kind, n = case["kind"], case["n"]

    def tet(r):
        return r**3, 6 * r**3, 0, 5 * (r - 1) ** 3

    def cloth(m):
        return m * m, 3 * m * m, 3 * m * m, 0

    if kind == "lattice":
        return n**3, (0, 0, 0, 0)
    if kind == "fill":
        return n, (0, 0, 0, 0)
    if kind == "mixed":
        return n**3, tuple(a + b for a, b in zip(tet(case["tet"]), cloth(case["cloth"])))
    if kind == "tet":
        return 0, tet(round(n ** (1 / 3)))
    if kind == "cloth":
        return 0, cloth(round(n**0.5))
    sizes, kinds = scenes.batch_sizes(n, case["layout"], case["lo"], case["hi"])
    share = min(1.0, case["tick"] / n) if kind == "serve" else 1.0
    fluid, solid = 0.0, [0.0] * 4
    for m, k in zip(sizes, kinds):
        if k == 0:
            fluid += share * m
        else:
            solid = [a + share * b for a, b in zip(solid, tet(round(m ** (1 / 3))) if k == 1 else cloth(round(m**0.5)))]
    return fluid, tuple(solid)


def work(case):
    if case["kind"] == "sort":
        return {"bytes": 16.0 * case["n"], "flops": 0.0}
    fluid, (solid, edges, dihedrals, tets) = _counts(case)
    rounds = case["substeps"] * case["iterations"]
    # state read and written, class and constraint records read once; the frames written once
    nbytes = 68.0 * (fluid + solid) + 16.0 * edges + 24.0 * dihedrals + 24.0 * tets
    # a neighbor pair in the density and delta sums, ~30 neighbors; a constraint's solve
    flops = rounds * (30.0 * 50.0 * fluid + 40.0 * edges + 150.0 * dihedrals + 120.0 * tets)
    if case.get("anisotropy"):
        nbytes += 48.0 * fluid
        flops += 30.0 * 40.0 * fluid
    if case.get("vorticity"):
        flops += case["substeps"] * 30.0 * 50.0 * fluid
    return {"bytes": float(nbytes), "flops": float(flops)}


# ---- the same step in 64 bits -------------------------------------------------------------------
def _walls(sc, x):
    """Signed distance to each static box and its outward normal: (n, walls), (n, walls, 3)."""
    c = torch.from_numpy(sc.colliders["center"]).to(x)
    he = torch.from_numpy(sc.colliders["half_extents"]).to(x)
    rel = x[:, None, :] - c
    off = rel - torch.minimum(torch.maximum(rel, -he), he)
    dist = off.norm(dim=2)
    depth, face = (he - rel.abs()).min(dim=2)
    inner = torch.zeros_like(off).scatter_(2, face[..., None], rel.gather(2, face[..., None]).sign())
    out = dist > 1e-6
    return torch.where(out, dist, -depth), torch.where(out[..., None], off / dist.clamp_min(1e-30)[..., None], inner)


def _pairs(x, h):
    """Ordered pairs (i, j) of particles in neighboring cells of size h that may come within h."""
    c = torch.floor(x / h).long()
    c = c - c.min(dim=0).values + 1
    d = c.max(dim=0).values + 2
    key = (c[:, 0] * d[1] + c[:, 1]) * d[2] + c[:, 2]
    key, order = torch.sort(key)
    at, found = torch.arange(len(x), device=x.device), []
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dz in (-1, 0, 1):
                k = key + (dx * d[1] + dy) * d[2] + dz
                lo, hi = torch.searchsorted(key, k), torch.searchsorted(key, k, right=True)
                m = hi - lo
                i = torch.repeat_interleave(at, m)
                j = lo[i] + torch.arange(len(i), device=x.device) - torch.repeat_interleave(m.cumsum(0) - m, m)
                i, j = order[i], order[j]
                ok = (i != j) & ((x[i] - x[j]).norm(dim=1) < 1.6 * h)
                found.append((i[ok], j[ok]))
    return torch.cat([f[0] for f in found]), torch.cat([f[1] for f in found])


def _exact_fluid(sc, case, x, v):
    m = {k: float(sc.fluid_mats[k][0]) for k in sc.fluid_mats.dtype.names}
    h, r, dt = m["smoothing_radius"], float(sc.radii[0]), float(np.float32(1 / 120)) / case["substeps"]
    k = 15.0 / (np.pi * h**3)
    rho, visc, cfl = max(m["rest_density"], 1.0), dt * m["viscosity"], m["cfl_radius"]

    def w(d):
        return torch.where(d < h, k * (1 - d / h) ** 2, 0.0)

    def dw(d):
        return torch.where(d < h, -2 * k * (1 - d / h) / h, 0.0)

    for _ in range(case["substeps"]):
        prev = x
        v = v + torch.tensor([0.0, float(np.float32(-9.81)), 0.0], dtype=x.dtype, device=x.device) * dt
        start = x + v * dt
        move = torch.zeros_like(start)
        a, b = _pairs(start, h)
        for it in range(case["iterations"]):
            s = start + move
            d = (s[a] - s[b]).norm(dim=1)
            near = d < h
            i, j, d = a[near], b[near], d[near]
            sd, wn = _walls(sc, s)
            gd = torch.where((sd >= 0) & (sd < h), 2 * sd, 2 * h)
            density = torch.zeros_like(s[:, 0]).index_add_(0, i, w(d)) + 0.12 * w(gd).sum(1)
            con = (density - rho).clamp_min(0.0) * m["density_constraint_scale"]
            live = d > 1e-6
            i, j, d = i[live], j[live], d[live]
            nrm = (s[i] - s[j]) / d[:, None]
            term = (-0.5 * (con[i] + con[j]) * dw(d))[:, None] * nrm
            if it > 0:
                rel = move[i] - move[j]
                term = term - (1 - 1 / (1 + visc * w(d)))[:, None] * rel
                proj = (rel * nrm).sum(1)
                term = term - torch.where(proj < -cfl, 0.5 * (cfl + proj), 0.0)[:, None] * nrm
            total = torch.zeros_like(s).index_add_(0, i, term)
            count = torch.zeros_like(s[:, 0]).index_add_(0, i, torch.ones_like(d))
            wall = ((-con[:, None] * torch.where(gd > 1e-6, dw(gd), 0.0))[..., None] * wn).sum(1)
            move = move + (0.7 * total + 0.08 * wall) / count.clamp_min(1.0)[:, None]
            y = start + move
            for _sweep in range(2):
                for q in range(sd.shape[1]):
                    one, n1 = (t[:, q] for t in _walls(sc, y))
                    y = y + n1 * (r - one).clamp_min(0.0)[:, None]
            move = y - start
        x = start + move
        v = (x - prev) / dt
        sd, wn = _walls(sc, x)
        sd, q = sd.min(1)
        n1 = wn[torch.arange(len(x), device=x.device), q]
        inward = (v * n1).sum(1).clamp_max(0.0)
        v = torch.where((sd <= r + 2.0e-3)[:, None], v - inward[:, None] * n1, v)
    return x, v


def _exact_soft(sc, case, x, v, w):
    dt, relax = float(np.float32(1 / 120)) / case["substeps"], 0.2

    def ids(a, *fields):
        return [torch.from_numpy(a[f].astype(np.int64)).to(x.device) for f in fields]

    def values(a, *fields):
        return [torch.from_numpy(a[f]).to(x) for f in fields]

    def cross(p, q):
        return torch.cross(p, q, dim=1)

    def dot(p, q):
        return (p * q).sum(1)

    def solve(x, verts, grads, C, lam, compliance, ok):
        # ok: the constraints that are not degenerate; the others do nothing
        alpha = compliance / dt**2
        den = sum(w[p] * dot(g, g) for p, g in zip(verts, grads)) + alpha
        dl = torch.where(ok & (den > 1e-6), -(C + alpha * lam) / den, 0.0)
        grads = [torch.where(ok[:, None], g, 0.0) for g in grads]
        y = x.clone()
        for p, g in zip(verts, grads):
            y.index_add_(0, p, (w[p] * dl * relax)[:, None] * g)
        return y, lam + dl

    e, d, t = sc.edges, sc.dihedrals, sc.tets
    for _ in range(case["substeps"]):
        prev = x
        v = v + torch.tensor([0.0, float(np.float32(-9.81)), 0.0], dtype=x.dtype, device=x.device) * dt
        x = x + v * dt
        le, ld, lt = (torch.zeros(len(a), dtype=x.dtype, device=x.device) for a in (e, d, t))
        for _it in range(case["iterations"]):
            if len(e):
                a, b = ids(e, "a", "b")
                rest, comp = values(e, "rest_length", "compliance")
                u = x[b] - x[a]
                length = u.norm(dim=1)
                u = u / length[:, None]
                x, le = solve(x, (a, b), (-u, u), length - rest, le, comp, length**2 > 1e-6)
            if len(d):
                e0, e1, o0, o1 = ids(d, "e0", "e1", "o0", "o1")
                rest, comp = values(d, "rest_angle", "compliance")
                edge = x[e1] - x[e0]
                n0, n1 = cross(x[e0] - x[o0], x[e1] - x[o0]), cross(x[e1] - x[o1], x[e0] - x[o1])
                length = edge.norm(dim=1)
                s0, s1 = n0 / dot(n0, n0)[:, None], n1 / dot(n1, n1)[:, None]
                f = [(dot(x[p] - x[q], edge) / length)[:, None] for p, q in ((o0, e1), (o1, e1), (e0, o0), (e0, o1))]
                g = (-(f[0] * s0 + f[1] * s1), -(f[2] * s0 + f[3] * s1), -length[:, None] * s0, -length[:, None] * s1)
                u0, u1 = n0 / n0.norm(dim=1, keepdim=True), n1 / n1.norm(dim=1, keepdim=True)
                theta = torch.atan2(dot(edge / length[:, None], cross(u0, u1)), dot(u0, u1))
                C = theta - rest
                C = C - 2 * np.pi * torch.floor((C + np.pi) / (2 * np.pi))
                ok = (length**2 > 1e-6) & (dot(n0, n0) > 1e-6) & (dot(n1, n1) > 1e-6)
                x, ld = solve(x, (e0, e1, o0, o1), g, C, ld, comp, ok)
            if len(t):
                p = [torch.from_numpy(t["p"][:, q].astype(np.int64)).to(x.device) for q in range(4)]
                rest, comp = values(t, "rest_volume", "compliance")
                p0, p1, p2, p3 = (x[q] for q in p)
                sv = dot(cross(p1 - p0, p2 - p0), p3 - p0) / 6
                f = (torch.where(sv >= 0, 1.0, -1.0).to(x) / 6)[:, None]
                g = (f * cross(p3 - p1, p2 - p1), f * cross(p2 - p0, p3 - p0), f * cross(p3 - p0, p1 - p0),
                     f * cross(p1 - p0, p2 - p0))
                x, lt = solve(x, p, g, sv.abs() - rest, lt, comp, torch.ones_like(sv, dtype=torch.bool))
        v = (x - prev) / dt
    return x, v


def exact(case, seed):
    """The step from the same inputs in 64 bits: a fluid lattice and the single soft bodies, from the
    uploaded state; the sorted pairs; None where the state was reached by steps, or is too large."""
    if case["kind"] == "sort":
        st = prepare(case, seed)
        k = st["keys"].long() & 0xFFFFFFFF
        k, o = torch.sort(k, stable=True)
        return k.to(torch.int32), st["idx"][o]
    if case["kind"] not in ("lattice", "cloth", "tet") or case["warm"]:
        return None
    sc = _scene(case, seed)
    if sc.n > EXACT_MOST:
        return None
    p = torch.from_numpy(sc.pos).cuda().double()
    v = torch.from_numpy(sc.vel).cuda().double()[:, :3]
    if case["kind"] == "lattice":
        x, v = _exact_fluid(sc, case, p[:, :3], v)
    else:
        x, v = _exact_soft(sc, case, p[:, :3], v, p[:, 3])
    return {"positions_inv_mass": torch.cat([x, p[:, 3:]], 1), "velocities": torch.cat([v, torch.zeros_like(v[:, :1])], 1)}
