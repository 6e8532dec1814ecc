"""Every form of a multigrid level at edge shapes: tiles with all smoothing
counts and the mixed form's FP32 levels against the oracle (one CG iteration from
x = 0 exposes one V-cycle), and the marching passes of small levels (a batch whose
cells add up takes them) bit for bit against the tiles of each case's own run."""
import numpy as np
import pytest

from ibmdem import cases
from ibmdem.abi import (BC_INFLOW, BC_OUTFLOW, BC_PERIODIC, BC_WALL, ERR_NOT_CONVERGED, FP64, K_MG_SMOOTH, MIXED,
                        Batch, IbmdemError, Simulation)

pytestmark = pytest.mark.gpu
P, W, I, O = BC_PERIODIC, BC_WALL, BC_INFLOW, BC_OUTFLOW

# one and two pairs per thread, rows in one tile and in several, partial tiles
# in every dimension, levels smaller than a halo, every side type
GRIDS = [
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
]


def _iterate(lib, n, bt, **kw):
    """One CG iteration from x = 0: one V-cycle applied to the right-hand side."""
    case = cases.build_case(*n, bt, rtol=1e-30, max_iter=1, **kw)
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


# tolerance as test_gpu_multigrid's: the rounding of two inner products
@pytest.mark.parametrize("pre,post", [(1, 1), (1, 2), (2, 1), (2, 3), (3, 2), (3, 4), (5, 5), (8, 6)])
@pytest.mark.parametrize("n,bt", [GRIDS[q] for q in (0, 2, 3, 5, 8, 9, 12)])
def test_smoothing_counts_in_tiles(gpu_lib, oracle_lib, n, bt, pre, post):
    kw = dict(mg_pre=pre, mg_post=post)
    _close(_iterate(gpu_lib, n, bt, **kw), _iterate(oracle_lib, n, bt, **kw), 1e-12)


def _visit_launches(lib, pre, post, precision):
    """Smoothing launches of one visit of level 0."""
    case = cases.build_case(48, 40, 56, [W] * 6, rtol=1e-30, max_iter=3, mg_pre=pre, mg_post=post, precision=precision)
    with Simulation(lib, case) as s:
        s.upload_poisson_rhs(np.random.default_rng(2).normal(size=(56, 40, 48)))
        s.profile_kernel(K_MG_SMOOTH)
        with pytest.raises(IbmdemError):
            s.poisson()
        return s.profile_read()[1] / 4   # z = M^-1 r at the start and in each iteration


# in tiles a launch for every two sweeps each way (marching passes would be one
# for each)
@pytest.mark.parametrize("pre,post,launches", [(2, 2, 2), (1, 1, 2), (3, 3, 4), (4, 4, 4), (7, 2, 5)])
def test_launches_of_a_visit_in_tiles(gpu_lib, pre, post, launches):
    assert _visit_launches(gpu_lib, pre, post, FP64) == launches


# the mixed form marches: a pass a sweep, but the last black and red ones apart
@pytest.mark.parametrize("pre,post,launches", [(2, 2, 5), (1, 1, 3), (3, 4, 8)])
def test_launches_of_a_mixed_visit(gpu_lib, pre, post, launches):
    assert _visit_launches(gpu_lib, pre, post, MIXED) == launches


# FP32 levels: a V-cycle commits about 8 roundings of 6e-8 in each of the 95
# half sweeps of its coarsest level and in fewer above it, 5e-5 of the scale
@pytest.mark.parametrize("pre,post", [(2, 2), (1, 1), (3, 2)])
@pytest.mark.parametrize("n,bt", GRIDS + [
    ((2, 2, 3), [W] * 6),             # the coarsest level alone, in all its forms
    ((11, 13, 14), [W, W, W, W, I, O]),
    ((3, 5, 7), [P] * 6),
    ((16, 16, 33), [P, P, P, P, W, W]),
    ((34, 27, 45), [W] * 6),
    ((49, 37, 21), [I, O, W, W, W, W]),
    ((25, 33, 19), [P, P, W, W, P, P]),
])
def test_mixed_levels(gpu_lib, oracle_lib, n, bt, pre, post):
    kw = dict(mg_pre=pre, mg_post=post)
    _close(_iterate(gpu_lib, n, bt, precision=MIXED, **kw), _iterate(oracle_lib, n, bt, **kw), 5e-5)


def _fluid(n, bt, precision, pre, post):
    inflow = [0.0, 0.0, 0.0]
    for d in range(3):
        if bt[2 * d] == I:
            inflow[d] = 0.05
    case = cases.build_case(*n, bt, visc=0.05, u_max=0.3, precision=precision, mg_pre=pre, mg_post=post,
                            inflow=tuple(inflow))
    mk, bd = cases.place_spheres(case, [])
    rng = np.random.default_rng(sum(n))
    f = [0.02 * rng.normal(size=n[::-1]) for _ in range(4)]
    for d in range(3):
        if bt[2 * d] == I:
            f[d] += 0.05
    return cases.Setup("fluid", case, mk, bd, f)


# with the large case's, the cells of levels 0 and 1 are more than tiles take,
# so every case marches there; in FP64 the small ones' own runs take tiles
@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("pre,post", [(2, 2), (1, 1), (3, 2), (2, 5)])
def test_small_levels_march_in_a_batch(gpu_lib, precision, pre, post):
    sets = [_fluid(n, bt, precision, pre, post) for n, bt in [((200, 200, 200), [W] * 6)] + GRIDS]
    with Batch(gpu_lib, [s.case for s in sets]) as b:
        for q, s in enumerate(sets):
            cases.load(b[q], s)
        infos = b.run(3)
        assert b.fused_solves() > 0
        got = [b[q].download_fields() for q in range(len(b))]
    for s, fields, info in list(zip(sets, got, infos))[1:]:
        with Simulation(gpu_lib, s.case) as one:
            cases.load(one, s)
            assert one.run(3).iterations == info.iterations
            for x, y in zip(fields, one.download_fields()):
                assert np.isfinite(x).all()
                np.testing.assert_array_equal(x, y)


# the mixed form keeps its level arrays in FP32 and no FP64 z beside them, except
# where there is one level: 8 n more there
def test_mixed_memory(gpu_lib):
    def memory(n, precision):
        with Simulation(gpu_lib, cases.build_case(*n, [W] * 6, precision=precision)) as s:
            return s.memory_bytes()
    n = (64, 64, 64)   # levels add up to less than 8/7 of level 0
    cells = 64 ** 3
    # FP64: z, r of every level, x and b of the coarser ones; mixed: x, b, r in FP32
    assert memory(n, FP64) - memory(n, MIXED) > cells * (8 + 8 * 1.14 + 16 * 0.14 - 12 * 1.15)
    one = (33, 35, 37)
    assert memory(one, MIXED) - memory(one, FP64) == 4 * 33 * 35 * 37   # 12 n + 8 n against 8 n + 8 n
