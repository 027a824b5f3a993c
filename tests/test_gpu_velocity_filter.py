"""The velocity filter (killApproachVelocity, newton.ts:238-303) at the sizes
where its sweep changes hands: fewer contact vertices than the dataflow
sweep's 64 lanes, exactly as many, a few more, several layers (edge pairs and
triangles that wait for each other), static partners (contacts with missing
cloth vertices), more contact vertices than fit its LDS (the round-based
sweep) and triangles that name a vertex twice (which only that one takes).  FP64 steps against the oracle, bit for bit: the sweep performs the
reference's operations in list order per vertex, so the bound is equality."""
import numpy as np
import pytest

import oracle_ffi as O
from closim_amd import _abi, mesh as M, scenes as S
from closim_amd.scene import DEFAULT_CONTACT_PARAMS, DEFAULT_MATERIAL, ContactSystem, create_scene
from closim_amd.solver import HipSolver
from contact_scenes import ALL

pytestmark = pytest.mark.gpu


def layers(nx, ny, count):
    """`count` sheets of 4 mm cells, 1.3 mm apart above the floor, sinking."""
    parts = [S.offset_mesh(nx, ny, 0.004 * nx, 0.004 * ny, 0.0, 0.0013 * (k + 1), 0.0) for k in range(count)]
    pos, uv, idx = S.merge_parts(parts)
    scene = create_scene(M.preprocess(pos, uv, idx, 0.15), DEFAULT_MATERIAL)
    rng = np.random.default_rng(nx * 100 + ny)
    scene.positions += rng.uniform(-1e-4, 1e-4, scene.positions.shape)
    scene.velocities.reshape(-1, 3)[:] = [0.01, -0.03, 0.0]
    scene.velocities += rng.uniform(-0.02, 0.02, scene.velocities.shape)
    scene.contact = ContactSystem(DEFAULT_CONTACT_PARAMS)
    scene.contact.setFloor(0.0)
    return scene


def check(make):
    sg, so = make(), make()
    g = HipSolver("fp64", newton_iters=1, pcg_max_iters=5)
    g.initialize(sg)
    o = O.OracleSolver(so, _abi.options(newton_iters=1, pcg_max_iters=5))
    g.step(1 / 60)
    o.step(1 / 60)
    assert np.array_equal(g.getPositions(), o.getPositions())
    assert np.array_equal(g.getVelocities(), o.getVelocities())
    return g.lastStats["contact"]


@pytest.mark.parametrize("nx,ny,count", [(1, 1, 1), (7, 7, 1), (12, 4, 1), (4, 5, 2), (9, 6, 2), (6, 6, 3), (63, 63, 1)])
def test_filter_matches_oracle(nx, ny, count):
    st = check(lambda: layers(nx, ny, count))
    assert st["active_pairs"] >= (nx + 1) * (ny + 1) // 2
    assert st["filter_rounds"] >= (2 if count > 1 else 1)


@pytest.mark.parametrize("name", ["plate", "crumpled"])
def test_filter_with_static_partners_and_folds(name):
    assert check(ALL[name])["active_pairs"] > 0


def with_repeated_corner(scene):
    """The scene with one more triangle, weightless, that names a vertex twice."""
    me = scene.mesh
    v, w = me.count - 10, me.count - 3
    me.indices = np.concatenate([me.indices, np.array([v, w, v], np.uint32)])
    me.inv_dm = np.concatenate([me.inv_dm, np.zeros(4, np.float32)])
    me.areas = np.concatenate([me.areas, np.zeros(1, np.float32)])
    me.tri_count += 1
    return scene


def sweep_without_stuck(ids, vals, v):
    """killApproachVelocity in list order, without the contacts that name a
    vertex twice and all that wait for them: what a sweep does that runs a
    contact once the earlier ones on its vertices have run."""
    stuck, left = set(), 0
    for (kind, p, a, b, c, d), val in zip(ids.tolist(), vals):
        w, nrm = val[:4], val[4:]
        vs = [p] if kind == 2 else [p, a, b, c] if kind == 0 else [a, b, c, d]
        if len(set(vs)) < len(vs) or stuck & set(vs):
            stuck |= set(vs)
            left += 1
            continue
        if kind == 2:
            v[p, 1] = max(v[p, 1], 0.0)
        elif kind == 0:
            t = w[0] * v[a] + w[1] * v[b] + w[2] * v[c]
            r = v[p] - t
            rel = r[0] * nrm[0] + r[1] * nrm[1] + r[2] * nrm[2]
            if rel < 0:
                j = -0.5 * rel
                v[p] += j * nrm
                for k, q in enumerate((a, b, c)):
                    v[q] -= j * w[k] * nrm
        else:
            r = (v[a] + v[b]) / 2 - (v[c] + v[d]) / 2
            rel = r[0] * nrm[0] + r[1] * nrm[1] + r[2] * nrm[2]
            if rel < 0:
                j = -0.25 * rel
                for q in (a, b):
                    v[q] += j * nrm
                for q in (c, d):
                    v[q] -= j * nrm
    return left


def test_triangle_that_names_a_vertex_twice():
    # the step ends, and every contact that waits for no such contact has run
    sc = with_repeated_corner(layers(6, 6, 2))
    x0 = sc.positions.copy()
    g = HipSolver("fp64", newton_iters=1, pcg_max_iters=5)
    g.initialize(sc)
    g.step(1 / 60)
    x1, v1 = g.getPositions().copy(), g.getVelocities().copy()
    assert np.isfinite(x1).all() and np.isfinite(v1).all()
    ids, vals, _ = g.probe_active_set(x0, x1)
    damp = 1 - min(max(DEFAULT_MATERIAL.damping, 0), 0.1)
    v = ((x1 - x0) / (1 / 60) * damp).reshape(-1, 3)
    left = sweep_without_stuck(ids, vals, v)
    print(f"{len(ids)} contacts, {left} left out", flush=True)
    assert 0 < left < len(ids)
    assert np.max(np.abs(v.reshape(-1) - v1)) <= 1e-12 * np.max(np.abs(v1))


@pytest.mark.parametrize("nx,ny,count", [(7, 7, 1), (9, 6, 2)])
def test_dataflow_sweep_that_gives_up_hands_over(nx, ny, count):
    # a bound of 0 ends the dataflow sweep before its first contact
    sg, so = layers(nx, ny, count), layers(nx, ny, count)
    g = HipSolver("fp64", newton_iters=1, pcg_max_iters=5)
    g.initialize(sg)
    o = O.OracleSolver(so, _abi.options(newton_iters=1, pcg_max_iters=5))
    assert not g.probe_filter_wait(0)
    for k in range(2):  # the second step does not try again
        g.step(1 / 60)
        o.step(1 / 60)
        assert g.probe_filter_wait(0xFFFFFFFF)
        assert np.array_equal(g.getPositions(), o.getPositions())
        assert np.array_equal(g.getVelocities(), o.getVelocities())
        assert 0 < g.lastStats["contact"]["filter_rounds"] <= g.lastStats["contact"]["active_pairs"]


def test_dataflow_sweep_does_not_give_up():
    g = HipSolver("fp64", newton_iters=1, pcg_max_iters=5)
    g.initialize(layers(9, 6, 3))
    g.step(1 / 60)
    assert not g.probe_filter_wait(0xFFFFFFFF)


def patches_on_floor_sheet(nx, k):
    """A floor sheet, and above its middle a patch of k x k cells: many
    contact vertices, and enough pairs that wait for each other."""
    parts = [S.offset_mesh(nx, nx, 0.004 * nx, 0.004 * nx, 0.0, 0.0013, 0.0),
             S.offset_mesh(k, k, 0.004 * k, 0.004 * k, 0.004 * (nx // 2) + 0.001, 0.0026, 0.004 * (nx // 2))]
    pos, uv, idx = S.merge_parts(parts)
    scene = create_scene(M.preprocess(pos, uv, idx, 0.15), DEFAULT_MATERIAL)
    rng = np.random.default_rng(nx)
    scene.positions += rng.uniform(-1e-4, 1e-4, scene.positions.shape)
    scene.velocities.reshape(-1, 3)[:] = [0.01, -0.03, 0.0]
    scene.velocities += rng.uniform(-0.02, 0.02, scene.velocities.shape)
    scene.contact = ContactSystem(DEFAULT_CONTACT_PARAMS)
    scene.contact.setFloor(0.0)
    return scene


@pytest.mark.parametrize("nx,k,lds", [(66, 5, True), (80, 8, False)])
def test_round_based_sweep_with_pairs_matches_oracle(nx, k, lds):
    # above the dataflow sweep's vertices, in LDS and beyond it: the contacts of
    # the sweep are the active set at the step's end
    sg, so = patches_on_floor_sheet(nx, k), patches_on_floor_sheet(nx, k)
    x0 = sg.positions.copy()
    g = HipSolver("fp64", newton_iters=1, pcg_max_iters=5)
    g.initialize(sg)
    o = O.OracleSolver(so, _abi.options(newton_iters=1, pcg_max_iters=5))
    g.step(1 / 60)
    o.step(1 / 60)
    x1, v1 = g.getPositions().copy(), g.getVelocities().copy()
    assert np.array_equal(x1, o.getPositions()) and np.array_equal(v1, o.getVelocities())
    rounds = g.lastStats["contact"]["filter_rounds"]
    ids, _, _ = g.probe_active_set(x0, x1)
    v = np.concatenate([ids[ids[:, 0] == 0][:, 1:5].ravel(), ids[ids[:, 0] == 1][:, 2:6].ravel(),
                        ids[ids[:, 0] == 2][:, 1]])
    nv, pairs = len(np.unique(v[v >= 0])), int((ids[:, 0] != 2).sum())
    need = nv * 32 + (len(ids) + 3) // 4 * 4  # velocities, lists and counters of the LDS form
    print(f"{nv} contact vertices, {len(ids)} contacts, {pairs} pairs, {rounds} rounds, {need} bytes", flush=True)
    assert nv > 4200  # beyond the dataflow sweep
    assert (need <= 160 * 1024 - 256) == lds and abs(need - 160 * 1024) > 4096
    assert pairs > 1000 and rounds > 1
