"""FP64 solves do not depend on the scale of the right-hand side: with
|b| ~ 1e-148 the squared residuals CG divides by fall below the smallest
normal number before the tolerance is met, and so they do with a tolerance
that no solve can meet."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

M = 0.1


@pytest.fixture(scope="module")
def hmc():
    from thirring2d_amd import hmc as H
    return H


def _setup(hmc, nt, nx):
    r = np.random.default_rng(17)
    lat = hmc.StaggeredLattice(nt, nx, m=M, g=0.5)
    lat.set_links(r.normal(size=(lat.V, 2)))
    return lat, r.normal(size=lat.V) + 1j * r.normal(size=lat.V)


# one workgroup, one to four sites per thread; whole and uneven regions
SIDES = [(16, 16), (16, 24), (24, 40), (40, 40), (64, 64), (96, 96)]


@pytest.mark.parametrize("nt, nx", SIDES)
@pytest.mark.parametrize("exponent", [-150, -148, -146, 140, 150])
def test_cg_fp64_scaled_rhs(hmc, nt, nx, exponent):
    """The scaled solve agrees with the unscaled one to the tolerance times the
    condition, 1e-10 (m^2 + 4) / m^2, twice, and in one workgroup takes its
    iterations within 2 % (the resident kernel ends a pass where its quotients
    leave the range, and the next one starts from there)."""
    lat, b = _setup(hmc, nt, nx)
    p = hmc.cg_params(tol_rel=1e-10)
    x0, i0 = lat.fmdm_invert_cg(b, p)
    x, i = lat.fmdm_invert_cg(b * 10.0 ** exponent, p)
    assert i0.status == 0 and i.status == 0
    if nt * nx <= 2048:
        assert i.restarts == i0.restarts
        assert abs(i.iterations - i0.iterations) <= i0.iterations // 50
    x = x / 10.0 ** exponent
    assert np.linalg.norm(x - x0) <= 2e-10 * (M * M + 4) / (M * M) * np.linalg.norm(x0)


@pytest.mark.parametrize("nt, nx", SIDES)
@pytest.mark.parametrize("tol", [1e-60, 1e-160])
def test_cg_fp64_unreachable_tolerance(hmc, nt, nx, tol):
    """The solve ends unconverged, with the solution at round-off: residuals
    of 1e-12 are met long before."""
    lat, b = _setup(hmc, nt, nx)
    x0, _ = lat.fmdm_invert_cg(b, hmc.cg_params(tol_rel=1e-12))
    x, i = lat.fmdm_invert_cg(b, hmc.cg_params(tol_rel=tol))
    assert i.status == -3 and i.true_rel_resid <= 1e-12
    assert np.linalg.norm(x - x0) <= 2e-12 * (M * M + 4) / (M * M) * np.linalg.norm(x0)
