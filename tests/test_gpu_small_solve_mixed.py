"""The mixed-precision inner solve in one launch (meshes of up to 64 HVP
tiles) against the separate kernels (CS_FLAG_EAGER): equal bit for bit, since
every product and every partial sum is formed by the same operations in the
same tree.  Sizes: one vertex group and its neighbours, one tile and more, the
largest meshes and the first beyond, vertices with more corners than the
entries kept in registers, every preconditioner and operator, caps."""
import numpy as np
import pytest

from closim_amd import _abi
from closim_amd.solver import HipSolver
from test_gpu_small_solve import fan, hung

pytestmark = pytest.mark.gpu
H = 1 / 60


def run(make, steps, **kw):
    g = HipSolver("mixed", **kw)
    g.initialize(make())
    its = []
    for _ in range(steps):
        g.step(H)
        its.append(g.lastStats["pcg_iters"])
    return g.getPositions().copy(), g.getVelocities().copy(), its


def check(make, steps=2, **kw):
    a = run(make, steps, **kw)
    b = run(make, steps, **dict(kw, flags=kw.get("flags", 0) | _abi.CS_FLAG_EAGER))
    assert a[2] == b[2]
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("nx,ny", [(1, 1), (12, 6), (15, 15), (15, 16), (16, 31), (19, 99), (62, 47)])
def test_sizes(nx, ny):
    check(lambda: hung(nx, ny))


@pytest.mark.parametrize("nx,ny", [(130, 89), (110, 139), (127, 127), (139, 139)])
def test_large_and_beyond(nx, ny):
    check(lambda: hung(nx, ny), steps=1, newton_iters=3)


@pytest.mark.parametrize("precond", [_abi.CS_PRECOND_JACOBI, _abi.CS_PRECOND_BLOCK_JACOBI])
@pytest.mark.parametrize("flags", [0, _abi.CS_FLAG_PSD_NEWTON, _abi.CS_FLAG_DEVICE_NEWTON])
def test_operators(precond, flags):
    check(lambda: hung(23, 17), precond=precond, flags=flags)


@pytest.mark.parametrize("k", [8, 9, 40])
def test_high_valence(k):
    check(lambda: fan(k))


@pytest.mark.parametrize("cap", [0, 1, 7, 9])
def test_caps(cap):
    check(lambda: hung(11, 13), pcg_max_iters=cap)
