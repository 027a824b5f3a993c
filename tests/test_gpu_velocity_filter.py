"""The velocity filter (killApproachVelocity, newton.ts:238-303) at the sizes
where its sweep changes hands: fewer contact vertices than the dataflow
sweep's 64 lanes, exactly as many, a few more, several layers (edge pairs and
triangles that wait for each other), static partners (contacts with missing
cloth vertices) and more contact vertices than fit its LDS (the round-based
sweep).  FP64 steps against the oracle, bit for bit: the sweep performs the
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
