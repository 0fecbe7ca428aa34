"""th2d_cg_last_kernel names the kernel that ran: the resident kernel takes
whole and uneven regions alike (th2d_cg_last_resident counts the whole ones)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STEP, RESIDENT, BOTH, SMALL = 0, 1, 2, 3


@pytest.fixture(scope="module")
def hmc():
    from thirring2d_amd import hmc as H
    return H


@pytest.fixture(scope="module")
def N():
    from thirring2d_amd import _native
    return _native


def _kernel(N, ctx):
    k = C.c_int(-1)
    N.check(N.lib().th2d_cg_last_kernel(ctx.ptr, C.byref(k)), "last_kernel")
    return k.value


def _batch(hmc, oracle, dims, seed=2300, m=0.1):
    lats, rest = [], []
    for k, (nt, nx) in enumerate(dims):
        r = np.random.default_rng(seed + k)
        A = r.normal(size=(nt * nx, 2))
        lat = hmc.StaggeredLattice(nt, nx, m=m, g=0.5)
        lat.set_links(A)
        lats.append(lat)
        rest.append((oracle.lattice(nt, nx, m=m, g=0.5), A,
                     r.normal(size=nt * nx) + 1j * r.normal(size=nt * nx)))
    return hmc.ChainBatch(lats), rest


def _check(oracle, rest, xs, infos, tol):
    for (L, A, b), x, inf in zip(rest, xs, infos):
        assert inf.status == 0
        r = b - oracle.fm_dag_mul(L, A, oracle.fm_mul(L, A, x))
        assert np.linalg.norm(r) <= 1.01 * tol * np.linalg.norm(b)


@pytest.mark.parametrize("dims", [
    [(96, 96)], [(96, 96), (96, 160)], [(70, 66), (2, 66), (206, 116)],  # uneven alone
    [(96, 96), (128, 128), (32, 32)], [(96, 64)], [(128, 128)],
])
@pytest.mark.parametrize("prec", [0, 2])
def test_resident_is_named(hmc, oracle, N, dims, prec):
    batch, rest = _batch(hmc, oracle, dims)
    tol = 1e-12 if prec == 0 else 1e-10
    xs, infos = batch.fmdm_invert_cg([b for _, _, b in rest],
                                     hmc.cg_params(tol_rel=tol, precision=prec))
    assert _kernel(N, batch.ctx) == RESIDENT
    _check(oracle, rest, xs, infos, tol)


def test_small_and_step_are_named(hmc, oracle, N):
    batch, rest = _batch(hmc, oracle, [(16, 16), (24, 40)])
    bs, ctx = [b for _, _, b in rest], batch.ctx
    batch.fmdm_invert_cg(bs, hmc.cg_params(tol_rel=1e-10))
    assert _kernel(N, ctx) == SMALL
    N.check(N.lib().th2d_set_cg_small(ctx.ptr, 0), "small")
    try:
        batch.fmdm_invert_cg(bs, hmc.cg_params(tol_rel=1e-10))
        assert _kernel(N, ctx) == STEP
    finally:
        N.lib().th2d_set_cg_small(ctx.ptr, 1)
    assert N.lib().th2d_cg_last_kernel(ctx.ptr, None) == N.TH2D_EARG
