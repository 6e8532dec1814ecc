"""Multigrid forms that depend on a level's size, against the CPU oracle:
one CG iteration from x = 0 exposes one V-cycle applied to the right-hand side
up to the rounding of two inner products, so the iterates agree to 1e-12 of
their scale (as in test_gpu_parity.test_one_preconditioned_iteration)."""
import numpy as np
import pytest

from ibmdem import cases
from ibmdem.abi import (BC_INFLOW, BC_OUTFLOW, BC_PERIODIC, BC_WALL, ERR_NOT_CONVERGED, IbmdemError, Batch, Simulation)

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


# the fused passes and transfers of the levels above the coarsest: one and two
# pairs per thread, whole and tiled rows, partial tiles and chunks in every
# dimension, levels smaller than a tile's halo, every side type
@pytest.mark.parametrize("n,bt", [
    ((4, 4, 4), [W] * 6),
    ((6, 4, 10), [P, P, P, P, W, W]),
    ((12, 20, 4), [W, W, P, P, P, P]),
    ((26, 14, 22), [P] * 6),
    ((62, 4, 8), [W] * 6),
    ((34, 58, 18), [W, W, W, W, I, O]),
    ((8, 130, 40), [P, P, W, W, P, P]),
    ((260, 28, 16), [P] * 6),
    ((264, 12, 20), [W] * 6),
    ((130, 44, 12), [I, O, P, P, W, W]),
    ((386, 8, 6), [P, P, W, W, W, W]),
    ((520, 30, 8), [I, O, W, W, P, P]),
    ((24, 40, 152), [W, W, I, O, P, P]),
])
def test_fused_passes(gpu_lib, oracle_lib, n, bt):
    _close(_iterate(gpu_lib, n, bt), _iterate(oracle_lib, n, bt), 1e-12)


@pytest.mark.parametrize("pre,post", [(1, 1), (1, 3), (3, 1), (4, 2)])
def test_smoothing_counts(gpu_lib, oracle_lib, pre, post):
    """Passes that are both first and last, and the buffers of odd counts."""
    n, bt = (40, 26, 36), [P, P, W, W, W, W]
    out = []
    for lib in (gpu_lib, oracle_lib):
        case = cases.build_case(*n, bt, rtol=1e-30, max_iter=1, mg_pre=pre, mg_post=post)
        rhs = np.random.default_rng(9).normal(size=n[::-1])
        with Simulation(lib, case) as s:
            s.upload_poisson_rhs(rhs)
            with pytest.raises(IbmdemError):
                s.poisson()
            out.append(s.download_poisson()[0])
    _close(out[0], out[1], 1e-12)


# the levels that one work-group runs: several pairs per thread, one, at most
# a wavefront's, and hierarchies of those alone; the same operations as one
# launch per operation, so equal bit for bit
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,bt", [
    ((32, 24, 40), [W] * 6),
    ((32, 32, 32), [P] * 6),
    ((36, 34, 26), [P, P, W, W, I, O]),
    ((48, 40, 36), [I, O, P, P, W, W]),
    ((16, 12, 20), [W, W, P, P, W, W]),
    ((8, 8, 16), [P, P, P, P, W, W]),
    ((4, 12, 6), [P] * 6),
])
def test_small_levels_in_one_work_group(gpu_lib, monkeypatch, n, bt, precision):
    out = []
    for separate in ("1", "0"):
        monkeypatch.setenv("IBMDEM_NO_TAIL", separate)
        out.append(_iterate(gpu_lib, n, bt, precision))
    assert np.abs(out[0]).max() > 0
    np.testing.assert_array_equal(out[0], out[1])


# levels whose prolongation is part of a smoothing pass: one pair per thread
# and two, rows in one tile and in several, chunks that begin in odd planes,
# coarse rows of odd length, every side type
@pytest.mark.parametrize("n,bt", [
    ((64, 118, 200), [W] * 6),
    ((130, 90, 78), [P, P, W, W, W, W]),
    ((130, 108, 110), [P] * 6),
    ((130, 100, 118), [W, W, P, P, I, O]),
    ((262, 90, 66), [I, O, W, W, P, P]),
    ((520, 60, 50), [P, P, W, W, W, W]),
])
def test_prolongation_in_a_pass(gpu_lib, oracle_lib, n, bt):
    _close(_iterate(gpu_lib, n, bt), _iterate(oracle_lib, n, bt), 1e-12)


# batches whose levels march where each case's own run takes tiles: several
# equal cases, uneven ones, and one that marches by itself among them
@pytest.mark.parametrize("sizes", [
    [(64, 48, 56)] * 6,
    [(96, 64, 40), (50, 80, 64), (72, 72, 64), (64, 36, 128)],
    [(32, 32, 32), (130, 90, 80), (48, 64, 32)],
])
def test_batch_marches_where_cases_tile(gpu_lib, sizes):
    setups = [cases.small_periodic(n=n, n_spheres=2) for n in sizes]

    def out(s):
        return s.download_fields()

    with Batch(gpu_lib, [s.case for s in setups]) as b:
        for q, s in enumerate(setups):
            cases.load(b[q], s)
        infos = b.run(3)
        got = [(out(b[q]), infos[q].iterations) for q in range(len(b))]
    for s, (fields, iterations) in zip(setups, got):
        with Simulation(gpu_lib, s.case) as one:
            cases.load(one, s)
            for _ in range(3):
                info = one.step()
            assert info.iterations == iterations
            for a, c in zip(fields, out(one)):
                np.testing.assert_array_equal(a, c)
