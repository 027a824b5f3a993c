"""The sorts of the contact lists at the sizes where they change kernels: one
work-group up to 16,384 pairs (whole rounds of 1,024 and one pair more), small
tiles beyond, large tiles from 2^17 pairs on.  A sheet lying on the floor has
one contact per vertex (four incidence pairs each).  A step with friction uses
the order of the active list, of the incidence and of the lagged-friction
table, so equality with the oracle checks all three; the order itself is
checked on the active set's records."""
import numpy as np
import pytest

from closim_amd.solver import HipSolver
from test_gpu_velocity_filter import check, layers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(15, 15), (15, 16), (31, 31), (31, 32), (63, 63), (63, 64)])
def test_step_matches_oracle(nx, ny):
    st = check(lambda: layers(nx, ny, 1))
    assert st["active_pairs"] > 0.4 * (nx + 1) * (ny + 1)


@pytest.mark.parametrize("nx,ny", [(127, 127), (127, 128), (255, 255), (369, 369)])
def test_active_list_is_sorted(nx, ny):
    sc = layers(nx, ny, 1)
    X = sc.positions.reshape(-1, 3)
    X[:, 1] = 0.001
    g = HipSolver("fp64")
    g.initialize(sc)
    ids, _, _ = g.probe_active_set(sc.positions, sc.positions, cap=(nx + 1) * (ny + 1))
    assert np.array_equal(ids[:, 1], np.arange((nx + 1) * (ny + 1)))  # (kind 2, vertex) in order
    assert np.all(ids[:, 0] == 2)
