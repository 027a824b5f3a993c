"""The FP64 inner solve in one launch (meshes of up to 64 work-groups of 64
vertices) and the gradient with 16 lanes per vertex, at the sizes where they
can go wrong: one work-group and one vertex more or less, the largest mesh and
the first beyond it, vertices with more corners than lanes, every
preconditioner and Hessian operator, few and many contacts.  Equality with the
oracle, and with the separate kernels, which CS_FLAG_TIMING selects: per-vertex
sums keep the reference's order and the reductions are correctly rounded."""
import numpy as np
import pytest

import oracle_ffi as O
from closim_amd import _abi, mesh as M, scenes as S
from closim_amd.scene import DEFAULT_CONTACT_PARAMS, DEFAULT_MATERIAL, ContactSystem, create_scene
from closim_amd.solver import HipBatch, HipSolver
from contact_scenes import ALL

pytestmark = pytest.mark.gpu
H = 1 / 60


def hung(nx, ny):
    """A sheet held by its first row, moving, its vertices jittered."""
    pos, uv, idx = M.build_grid(nx, ny, 0.01 * nx, 0.01 * ny)
    scene = create_scene(M.preprocess(pos, uv, idx, 0.15), DEFAULT_MATERIAL)
    rng = np.random.default_rng(nx * 1000 + ny)
    scene.positions += rng.uniform(-1e-4, 1e-4, scene.positions.shape)
    scene.velocities += rng.uniform(-0.1, 0.1, scene.velocities.shape)
    for i in range(nx + 1):
        scene.pinned[i] = tuple(float(c) for c in scene.positions[3 * i:3 * i + 3])
    return scene


def fan(k):
    """k triangles around one vertex, and a second ring: valences up to k."""
    a = 2 * np.pi * np.arange(k) / k
    ring = np.stack([np.cos(a), np.zeros(k), np.sin(a)], 1)
    P = np.concatenate([[[0, 0, 0]], 0.05 * ring, 0.1 * ring]).astype(np.float32)
    idx = []
    for i in range(k):
        j = (i + 1) % k
        idx += [0, 1 + i, 1 + j, 1 + i, 1 + k + i, 1 + j, 1 + j, 1 + k + i, 1 + k + j]
    uv = P[:, [0, 2]].copy()
    scene = create_scene(M.preprocess(P.reshape(-1), uv.reshape(-1), np.array(idx, np.uint32), 0.15), DEFAULT_MATERIAL)
    rng = np.random.default_rng(k)
    scene.positions += rng.uniform(-1e-3, 1e-3, scene.positions.shape)
    scene.pinned[1] = tuple(float(c) for c in scene.positions[3:6])
    return scene


def step(make, **kw):
    g = HipSolver("fp64", **kw)
    g.initialize(make())
    g.step(H)
    return g.getPositions().copy(), g.getVelocities().copy(), g.lastStats["pcg_iters"]


def check(make, oracle=True, **kw):
    x, v, its = step(make, **kw)
    xs, vs, its_s = step(make, **dict(kw, flags=kw.get("flags", 0) | _abi.CS_FLAG_TIMING))
    assert its == its_s
    assert np.array_equal(x, xs) and np.array_equal(v, vs)
    if oracle:
        o = O.OracleSolver(make(), _abi.options(**kw))
        o.step(H)
        assert np.array_equal(x, o.getPositions()) and np.array_equal(v, o.getVelocities())


@pytest.mark.parametrize("nx,ny", [(1, 1), (8, 6), (7, 7), (12, 4), (15, 7), (10, 11)])
def test_sizes_match_oracle(nx, ny):
    check(lambda: hung(nx, ny))


@pytest.mark.parametrize("nx,ny", [(62, 64), (63, 63), (63, 64)])
def test_largest_and_first_beyond_match_separate_kernels(nx, ny):
    check(lambda: hung(nx, ny), oracle=False, newton_iters=3)


@pytest.mark.parametrize("precond", [_abi.CS_PRECOND_JACOBI, _abi.CS_PRECOND_BLOCK_JACOBI])
@pytest.mark.parametrize("hvp", [_abi.CS_HVP_FD, _abi.CS_HVP_ANALYTIC])
def test_operators_match_oracle(precond, hvp):
    check(lambda: hung(13, 9), precond=precond, hvp_mode=hvp)


def test_psd_operator_matches_separate_kernels():
    check(lambda: hung(13, 9), oracle=False, hvp_mode=_abi.CS_HVP_ANALYTIC, flags=_abi.CS_FLAG_PSD_NEWTON)


@pytest.mark.parametrize("k", [7, 8, 9, 16, 17, 40])
def test_high_valence_matches_oracle(k):
    check(lambda: fan(k))


@pytest.mark.parametrize("cap", [0, 1, 2])
def test_iteration_caps(cap):
    check(lambda: hung(9, 9), pcg_max_iters=cap)


@pytest.mark.parametrize("name", ["floor", "plate", "crumpled", "stacked"])
def test_contacts_match_oracle(name):
    check(ALL[name])


@pytest.mark.parametrize("nx,ny", [(180, 180), (180, 181)])
def test_gradient_on_both_sides_of_its_rule(nx, ny):
    # 32,761 and 32,942 vertices; one Newton iteration with one PCG iteration
    def make():
        return hung(nx, ny)
    x, v, _ = step(make, newton_iters=1, pcg_max_iters=1)
    o = O.OracleSolver(make(), _abi.options(newton_iters=1, pcg_max_iters=1))
    o.step(H)
    assert np.array_equal(x, o.getPositions()) and np.array_equal(v, o.getVelocities())


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_more_solves_at_once_than_tickets(precision):
    # six meshes of 64 work-groups each, four of which fit 256 compute units:
    # whoever gets no ticket takes the separate kernels, with the same results
    nx, ny = (62, 64) if precision == "fp64" else (110, 139)
    kw = dict(newton_iters=3)
    alone = HipSolver(precision, **kw)
    alone.initialize(hung(nx, ny))
    gs = [HipSolver(precision, **kw) for _ in range(6)]
    for g in gs:
        g.initialize(hung(nx, ny))
    B = HipBatch(gs, threads=6)
    for _ in range(2):
        alone.step(H)
        assert B.step(H) == [0] * 6
        for g in gs:
            assert np.array_equal(g.getPositions(), alone.getPositions())
            assert np.array_equal(g.getVelocities(), alone.getVelocities())
    for g in gs:
        g.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nx,ny", [(1, 1), (13, 9), (40, 30)])
def test_solve_that_gives_up_hands_over(precision, nx, ny):
    # a bound of 0 polls ends the first exchange of every work-group: the
    # separate kernels solve from the same inputs and no later solve tries again
    a, b = HipSolver(precision), HipSolver(precision, flags=_abi.CS_FLAG_TIMING)
    a.initialize(hung(nx, ny))
    b.initialize(hung(nx, ny))
    assert not a.probe_exchange_wait(0)
    for _ in range(2):
        a.step(H)
        b.step(H)
        assert a.probe_exchange_wait(0xFFFFFFFF)
        assert a.lastStats["pcg_iters"] == b.lastStats["pcg_iters"]
        assert np.array_equal(a.getPositions(), b.getPositions())
        assert np.array_equal(a.getVelocities(), b.getVelocities())
    c = HipSolver(precision)
    c.initialize(hung(nx, ny))
    c.step(H)
    assert not c.probe_exchange_wait(0xFFFFFFFF)


def grid_below(nx, fine):
    """A sheet sinking on the floor, one vertex of it just above a static grid
    of fine x fine points, 2 mm from its middle to its sides."""
    pos, uv, idx = S.merge_parts([S.offset_mesh(nx, nx, 0.004 * nx, 0.004 * nx, 0.0, 0.0013, 0.0)])
    scene = create_scene(M.preprocess(pos, uv, idx, 0.15), DEFAULT_MATERIAL)
    scene.positions += np.random.default_rng(nx).uniform(-1e-4, 1e-4, scene.positions.shape)
    scene.velocities.reshape(-1, 3)[:] = [0.01, -0.03, 0.0]
    X = scene.positions.reshape(-1, 3)
    p = X[(nx // 2) * (nx + 1) + nx // 2]
    at = np.linspace(-0.002, 0.002, fine)
    V = np.array([[p[0] + a, p[1] - 0.001, p[2] + b] for a in at for b in at], np.float32)
    q = [a * fine + b for a in range(fine - 1) for b in range(fine - 1)]
    T = [t for k in q for t in ([k, k + 1, k + fine], [k + 1, k + fine + 1, k + fine])]
    scene.contact = ContactSystem(DEFAULT_CONTACT_PARAMS)
    scene.contact.setFloor(0.0)
    scene.contact.setStaticMesh(V.reshape(-1), np.array(T, np.uint32).reshape(-1))
    return scene


@pytest.mark.parametrize("fine,one_launch", [(2, True), (3, False), (6, False)])
def test_rule_looks_at_the_vertex_with_the_most_contacts(fine, one_launch):
    # few contacts a vertex on average, but some 50, 270 and 1,900 on one
    kw = dict(newton_iters=2)
    check(lambda: grid_below(12, fine), **kw)
    g = HipSolver("fp64", **kw)
    sc = grid_below(12, fine)
    g.initialize(sc)
    ids, _, _ = g.probe_active_set(sc.positions, sc.positions)
    v = np.concatenate([ids[ids[:, 0] == 0][:, 1:5].ravel(), ids[ids[:, 0] == 1][:, 2:6].ravel(),
                        ids[ids[:, 0] == 2][:, 1]])
    most = np.bincount(v[v >= 0]).max()
    print(f"most entries of a vertex {most}", flush=True)
    assert (most <= 64) == one_launch
    g.probe_exchange_wait(0)  # the one-launch solve, where it is tried, gives up at once
    g.step(H)
    assert g.probe_exchange_wait(0xFFFFFFFF) == one_launch


@pytest.mark.parametrize("fine,groups", [(5, False), (6, True), (9, True)])
def test_contact_sums_on_both_sides_of_their_rule(fine, groups):
    # 15 and 25 entries a vertex on average, 1,100 to 4,800 on one: the sums by a
    # thread per component and by a work-group (in several rounds of 256)
    kw = dict(newton_iters=2)
    sc = grid_below(12, fine)
    g = HipSolver("fp64", **kw)
    g.initialize(sc)
    ids, _, _ = g.probe_active_set(sc.positions, sc.positions)
    v = np.concatenate([ids[ids[:, 0] == 0][:, 1:5].ravel(), ids[ids[:, 0] == 1][:, 2:6].ravel(),
                        ids[ids[:, 0] == 2][:, 1]])
    n = np.bincount(v[v >= 0])
    print(f"{n.sum()} entries, {(n > 0).sum()} vertices, {n.max()} on one", flush=True)
    assert (n.sum() >= 16 * (n > 0).sum()) == groups and n.max() > 512
    g.step(H)
    o = O.OracleSolver(grid_below(12, fine), _abi.options(**kw))
    o.step(H)
    assert np.array_equal(g.getPositions(), o.getPositions()) and np.array_equal(g.getVelocities(), o.getVelocities())
