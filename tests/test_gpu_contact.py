"""The contact scan's two forms (32 lanes a marker, one thread a marker) against
the oracle bit for bit: few and many scanning markers per block, more
candidates in a row of cells or in all than the first form holds, rows that
wrap in x, walls."""
import numpy as np
import pytest

from ibmdem import cases
from ibmdem.abi import BC_PERIODIC, BC_WALL, Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("markers", [40, 201, 900, 4000])
@pytest.mark.parametrize("walls", [False, True])
def test_contact_scan_forms(gpu_lib, oracle_lib, markers, walls):
    n = (24, 20, 22)
    case = cases.build_case(*n, [BC_WALL if walls else BC_PERIODIC] * 6, visc=0.05, kn_coeff=1e5, restitution=0.9,
                            u_max=0.3, max_pairs=2000)
    # shells overlap along x, also across the periodic face, and along z
    cs = [(4.2, 9.8, 4.1), (12.1, 9.7, 4.4), (20.0, 9.9, 4.2), (12.3, 10.1, 12.0)]
    mk, bd = cases.place_spheres(case, [cases.Sphere(c, 8.0, 2.0, markers) for c in cs])
    rng = np.random.default_rng(4)
    mk.v[:] = rng.normal(0.0, 0.02, size=mk.v.shape)
    out = []
    for lib in (gpu_lib, oracle_lib):
        with Simulation(lib, case) as s:
            s.upload_bodies(bd)
            s.upload_markers(mk)
            s.contact()
            out.append(s.download_markers().fcol)
    assert np.abs(out[1]).max() > 0
    np.testing.assert_array_equal(out[0], out[1])


# the bodies in reach: fewer and more bodies than a block and than a chunk of
# either length, several in reach at once and across a periodic side, and none
@pytest.mark.parametrize("bodies", [2, 17, 65, 130, 4097, 4160])
def test_bodies_in_reach(gpu_lib, oracle_lib, bodies):
    n = (40, 36, 44)
    case = cases.build_case(*n, [BC_PERIODIC] * 4 + [BC_WALL] * 2, visc=0.05, kn_coeff=1e5, restitution=0.9, u_max=0.3,
                            max_pairs=500)
    rng = np.random.default_rng(bodies)
    cs = [tuple(c) for c in rng.uniform(1.5, np.array(n) - 1.5, (bodies, 3))]
    mk, bd = cases.place_spheres(case, [cases.Sphere(c, 1.0, 2.0, 3) for c in cs])
    out = []
    for lib in (gpu_lib, oracle_lib):
        with Simulation(lib, case) as s:
            s.upload_bodies(bd)
            s.upload_markers(mk)
            s.contact()
            out.append(s.download_markers().fcol)
    assert bodies < 100 or np.abs(out[1]).max() > 0
    np.testing.assert_array_equal(out[0], out[1])


# shells denser than the first form holds in some blocks and not in others, and
# blocks where some of the scanning markers fit and the rest do not
@pytest.mark.parametrize("markers", [(2000, 2000), (4000, 201), (60, 6000), (1000, 3000)])
def test_contact_scan_overflow(gpu_lib, oracle_lib, markers):
    case = cases.build_case(40, 36, 34, [BC_PERIODIC] * 6, visc=0.05, kn_coeff=1e5, restitution=0.9, u_max=0.3,
                            max_pairs=4000)
    cs = [(8.2, 17.8, 17.1), (20.6, 17.7, 17.4)]
    mk, bd = cases.place_spheres(case, [cases.Sphere(c, 12.0, 2.0, m) for c, m in zip(cs, markers)])
    mk.v[:] = np.random.default_rng(6).normal(0.0, 0.02, size=mk.v.shape)
    out = []
    for lib in (gpu_lib, oracle_lib):
        with Simulation(lib, case) as s:
            s.upload_bodies(bd)
            s.upload_markers(mk)
            s.contact()
            out.append(s.download_markers().fcol)
    assert np.abs(out[1]).max() > 0
    np.testing.assert_array_equal(out[0], out[1])


# several scanning markers one after the other on the same lanes, each with
# another number of candidates than the one before it (none among them)
@pytest.mark.parametrize("seed", [1, 2])
def test_contact_scan_turns(gpu_lib, oracle_lib, seed):
    case = cases.build_case(30, 28, 26, [BC_PERIODIC] * 6, visc=0.05, kn_coeff=1e5, restitution=0.9, u_max=0.3,
                            max_pairs=500)
    rng = np.random.default_rng(seed)
    cs = [tuple(c) for c in rng.uniform(0.0, 26.0, (40, 3))]
    mk, bd = cases.place_spheres(case, [cases.Sphere(c, 5.0, 2.0, 30 + q) for q, c in enumerate(cs)])
    mk.v[:] = rng.normal(0.0, 0.02, size=mk.v.shape)
    out = []
    for lib in (gpu_lib, oracle_lib):
        with Simulation(lib, case) as s:
            s.upload_bodies(bd)
            s.upload_markers(mk)
            s.contact()
            out.append(s.download_markers().fcol)
    assert np.abs(out[1]).max() > 0
    np.testing.assert_array_equal(out[0], out[1])
