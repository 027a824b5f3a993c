"""The FP64 Schwarz apply (applySchwarz, schwarz.ts:255-309) at the edges of
its kernel: rows that fill a multiple of 64 exactly and one vertex less or
more, full and partial domains side by side in one wave, an odd number of
domains, single-vertex domains, the widest instance, and a Jacobi-fallback
domain beside a factored one.  Equality with the oracle: the apply performs
the reference's operations in its order."""
import numpy as np
import pytest

import oracle_ffi as O
from closim_amd import _abi, scenes as S
from closim_amd.solver import HipSolver

pytestmark = pytest.mark.gpu


def check(make, sizes, seed, diag_of=None):
    sc = make()
    rng = np.random.default_rng(seed)
    x = sc.positions * 1.02 + 1e-4 * rng.standard_normal(sc.positions.shape)
    diag = np.repeat(np.asarray(sc.mesh.masses, np.float64), 3) * 3600.0 + 50.0 * (1 + rng.random(len(x)))
    o = O.OracleSolver(make())
    if diag_of:
        diag = diag_of(diag, o.schwarz_domains(*sizes)[0])
    r = rng.standard_normal(len(x))
    g = HipSolver("fp64", precond=_abi.CS_PRECOND_SCHWARZ, schwarz=sizes)
    g.initialize(make())
    z64, _, flags, _ = g.probe_schwarz(x, diag, r)
    zo, fo = o.schwarz_apply(x, diag, r, *sizes)
    assert np.array_equal(flags, fo)
    assert np.array_equal(z64, zo)
    return fo


@pytest.mark.parametrize("target", [1, 2, 20, 21, 22, 42, 43, 63, 64, 65, 85, 86, 107, 128, 149, 170])
def test_apply_matches_oracle(target):
    assert np.all(check(S.strip_pull, (target, 1, target), target) == 1)


def test_fallback_beside_factored_domains():
    def break_some(diag, dom):
        # every third domain's diagonal far below its stiffness
        out = diag.copy()
        out[np.repeat(dom % 3 == 0, 3)] = -1e9
        return out
    flags = check(S.strip_pull, (64, 1, 64), 5, break_some)
    assert 0 < flags.sum() < len(flags)
