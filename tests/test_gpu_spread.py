"""The spread's forms of the weights' 1/dV against the oracle: folded into
fdrag*vol exactly (power-of-two spacing), by one division per entry (FP64), or
divided weight by weight (mixed); markers whose supports cross tile edges,
periodic faces and walls, in lists of less than one to several staged chunks.
Tolerance as test_gpu_parity.test_spread_and_mdf_update: a few roundings of
each cell's largest term."""
import numpy as np
import pytest

from ibmdem import cases
from ibmdem.abi import BC_PERIODIC, BC_WALL, Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,precision", [(1.0, 0), (0.5, 1), (0.3, 0), (0.3, 1)])
@pytest.mark.parametrize("walls", [False, True])
def test_spread_forms(gpu_lib, oracle_lib, h, precision, walls):
    n = (20, 17, 24)
    bt = [BC_WALL if walls else BC_PERIODIC] * 6
    case = cases.build_case(*n, bt, h=h, visc=0.05, dt=0.1, precision=precision)
    cs = [(5.2, 4.6, 4.4), (5.4, 12.9, 4.1), (14.8, 8.3, 12.2), (14.1, 8.7, 19.6)]
    mk, bd = cases.place_spheres(case, [cases.Sphere(tuple(h * x for x in c), 7.0 * h, 1.5, m)
                                        for c, m in zip(cs, (9, 150, 300, 40))], h)
    rng = np.random.default_rng(3)
    mk.v[:] = rng.normal(size=mk.v.shape)
    u = [rng.normal(size=n[::-1]) for _ in range(3)]
    out = []
    for lib in (gpu_lib, oracle_lib):
        with Simulation(lib, case) as s:
            s.upload_bodies(bd)
            s.upload_markers(mk)
            s.upload_fields(*u, None)
            s.begin_step()
            for _ in range(2):
                s.interpolate()
                s.spread()
            out.append((s.download_force(), s.download_fields()[:3]))
    for a, b in zip(out[0][0] + out[0][1], out[1][0] + out[1][1]):
        assert np.abs(b).max() > 0
        assert np.abs(a - b).max() < 1e-14 * np.abs(b).max()


# staged chunks that are images throughout, in one, two and three dimensions:
# their rows are written by all lanes and then overwritten in part by the lane
# that stages the entry
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("h", [1.0, 0.3])
@pytest.mark.parametrize("bt", [[BC_PERIODIC] * 6, [BC_WALL] * 6, [BC_PERIODIC] * 2 + [BC_WALL] * 2 + [BC_PERIODIC] * 2])
def test_spread_of_images(gpu_lib, oracle_lib, bt, h, precision):
    n = (16, 24, 17)
    case = cases.build_case(*n, bt, h=h, visc=0.05, dt=0.1, precision=precision)
    lo, hi = 1.4, [m - 1.4 for m in n]
    cs = [(x, y, z) for z in (lo, hi[2]) for y in (lo, hi[1]) for x in (lo, hi[0])]   # corners
    cs += [(lo, 12.0, hi[2]), (8.0, lo, 8.5), (8.0, 12.0, hi[2])]                     # an edge and faces
    mk, bd = cases.place_spheres(case, [cases.Sphere(tuple(h * x for x in c), 2.4 * h, 1.5, 40 + 9 * q)
                                        for q, c in enumerate(cs)], h)
    rng = np.random.default_rng(8)
    mk.v[:] = rng.normal(size=mk.v.shape)
    u = [rng.normal(size=n[::-1]) for _ in range(3)]
    out = []
    for lib in (gpu_lib, oracle_lib):
        with Simulation(lib, case) as s:
            s.upload_bodies(bd)
            s.upload_markers(mk)
            s.upload_fields(*u, None)
            s.begin_step()
            s.interpolate()
            s.spread()
            out.append((s.download_force(), s.download_fields()[:3]))
    for a, b in zip(out[0][0] + out[0][1], out[1][0] + out[1][1]):
        assert np.abs(b).max() > 0
        assert np.abs(a - b).max() < 1e-13 * np.abs(b).max()
