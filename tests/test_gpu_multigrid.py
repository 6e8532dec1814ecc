"""Multigrid forms that depend on a level's size, against the CPU oracle:
one CG iteration from x = 0 exposes one V-cycle applied to the right-hand side
up to the rounding of two inner products, so the iterates agree to 1e-12 of
their scale (as in test_gpu_parity.test_one_preconditioned_iteration)."""
import numpy as np
import pytest

from ibmdem import cases
from ibmdem.abi import (BC_INFLOW, BC_OUTFLOW, BC_PERIODIC, BC_WALL, ERR_NOT_CONVERGED, IbmdemError, Simulation)

pytestmark = pytest.mark.gpu
P, W, I, O = BC_PERIODIC, BC_WALL, BC_INFLOW, BC_OUTFLOW


def _iterate(lib, n, bt, precision=0):
    case = cases.build_case(*n, bt, rtol=1e-30, max_iter=1, precision=precision)
    rhs = np.random.default_rng(5).normal(size=n[::-1])
    rhs -= rhs.mean()
    with Simulation(lib, case) as s:
        s.upload_poisson_rhs(rhs)
        with pytest.raises(IbmdemError) as e:
            s.poisson()
        assert e.value.code == ERR_NOT_CONVERGED
        return s.download_poisson()[0]


def _close(a, b, tol):
    assert np.abs(b).max() > 0
    assert np.abs(a - b).max() < tol * np.abs(b).max()


# the coarsest level in one work-group (a few cells to the largest that fits,
# odd row lengths, both smoothers), and in tiles (one tile and less in a
# dimension, partial tiles, several tiles, wrapped halos)
@pytest.mark.parametrize("n,bt", [
    ((2, 2, 3), [W] * 6),
    ((7, 5, 9), [W] * 6),
    ((8, 13, 9), [P, P, W, W, W, W]),
    ((11, 13, 14), [W, W, W, W, I, O]),
    ((13, 27, 21), [W] * 6),
    ((16, 16, 33), [P, P, P, P, W, W]),
    ((32, 15, 17), [P, P, W, W, W, W]),
    ((15, 23, 21), [I, O, W, W, P, P]),
    ((3, 5, 7), [P] * 6),
    ((9, 8, 7), [P] * 6),
    ((21, 13, 30), [W, W, P, P, W, W]),
    ((25, 21, 18), [P] * 6),
    ((34, 27, 45), [W] * 6),
    ((6, 10, 161), [P, P, P, P, W, W]),
    ((49, 37, 21), [I, O, W, W, W, W]),
    ((25, 33, 19), [P, P, W, W, P, P]),
])
def test_coarsest_level_forms(gpu_lib, oracle_lib, n, bt):
    _close(_iterate(gpu_lib, n, bt), _iterate(oracle_lib, n, bt), 1e-12)
