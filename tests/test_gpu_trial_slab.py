"""Trial validation's slab between the triangles of a pair: steps whose
triangles invert, thin out or coincide, far from the origin and in two fast
layers, against the oracle, with the smallest distance and time of impact that
the skipped pairs must not change.  They are minima of the same rounded values,
so they are equal; positions keep the 1e-9 of the other contact trajectories."""
import numpy as np
import pytest

import oracle_ffi as O
from closim_amd import _abi, scenes as S
from closim_amd.solver import HipSolver
from contact_scenes import stacked_patches

pytestmark = pytest.mark.gpu
H = 1.0 / 60.0
NX = 6
SIDE = 0.1 / NX  # of a grid cell of the patch


def scene_of(name):
    rng = np.random.default_rng(5)
    scene = stacked_patches() if name == "layers" else S.floor_patch(nx=NX, hover=2e-3)
    X = scene.positions.reshape(-1, 3)
    V = scene.velocities.reshape(-1, 3)
    if name == "rough":  # half a cell a step and vertex: triangles invert on the way
        X += rng.normal(0, 0.1 * SIDE, X.shape)
        X[:, 1] += 0.5 * SIDE
        V += rng.normal(0, 0.5 * SIDE / H, V.shape)
    elif name == "sliver":  # rows 1e-7 of a cell off the line of their neighbours
        g = X.reshape(NX + 1, NX + 1, 3)
        g[2] = g[1] + 1e-7 * SIDE
        V += rng.normal(0, 0.05 * SIDE / H, V.shape)
    elif name == "coincident":  # zero-length edges: no weight may be 0/0 unseen
        X[NX + 4] = X[NX + 3]
        X[3] = X[2]
        V += rng.normal(0, 0.05 * SIDE / H, V.shape)
    elif name == "far":  # positions rounded to 1e-9 of a cell
        X[:, 0] += 1e5
    else:  # the layers meet within the step
        V[: len(V) // 2, 1] = 0.3
        V[len(V) // 2 :, 1] = -0.3
        V += rng.normal(0, 0.02, V.shape)
    return scene


def bits(a):
    return np.float64(a).tobytes()


@pytest.mark.parametrize("name", ["rough", "sliver", "coincident", "far", "layers"])
def test_steps_judged_as_the_oracle_judges(name):
    g = HipSolver("fp64")
    g.initialize(scene_of(name))
    o = O.OracleSolver(scene_of(name), _abi.options())
    rejected = 0
    for k in range(3):
        g.step(H)
        o.step(H)
        cg, co = g.lastStats["contact"], o.lastStats["contact"]
        print(f"{name} step {k}: {cg}", flush=True)
        a, b = g.getPositions(), o.getPositions()
        assert np.max(np.abs(a - b)) <= 1e-9 * np.max(np.abs(b))
        for key in ("candidate_pairs", "active_pairs", "rejected_line_search_steps", "ccd_failures"):
            assert cg[key] == co[key], (k, key)
        for key in ("min_distance", "min_toi"):
            assert bits(cg[key]) == bits(co[key]), (k, key, cg[key], co[key])
        rejected += cg["rejected_line_search_steps"]
    assert rejected > 0 or name in ("far", "rough")  # the others reach a rejection
