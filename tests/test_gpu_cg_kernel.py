"""th2d_cg_last_kernel names the kernel that ran: the resident kernel takes
whole and uneven regions alike (th2d_cg_last_resident counts the whole ones),
and the step kernel's graph, the timeout of an FP64 solve and the fused MD
steps are reached on purpose here."""
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


def _fallbacks(N, ctx):
    n = C.c_long()
    N.check(N.lib().th2d_cg_sync_fallbacks(ctx.ptr, C.byref(n)), "fallbacks")
    return n.value


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
    [(96, 96), (100, 70), (48, 130), (66, 66)] * 16,         # every XCD full, FP64 in two launches
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


@pytest.mark.parametrize("prec", [0, 2])
def test_step_graph_matches_eager(hmc, oracle, N, prec):
    """The step kernel's launches as replays of a captured graph and one by
    one, bitwise alike over three solves with other work between them."""
    dims = [(96, 96), (40, 56), (96, 160)]
    batch, rest = _batch(hmc, oracle, dims)
    ctx = batch.ctx
    rng = np.random.default_rng(8)
    rhs = [[rng.normal(size=nt * nx) + 1j * rng.normal(size=nt * nx) for nt, nx in dims]
           for _ in range(3)]
    out = {}
    N.check(N.lib().th2d_set_cg_resident(ctx.ptr, 0), "resident")
    try:
        for on in (1, 0):
            N.check(N.lib().th2d_set_cg_graph(ctx.ptr, on), "graph")
            out[on] = []
            for b in rhs:
                out[on].append(batch.fmdm_invert_cg(b, hmc.cg_params(tol_rel=1e-10, precision=prec)))
                assert _kernel(N, ctx) == STEP
    finally:
        N.lib().th2d_set_cg_graph(ctx.ptr, 0)
        N.lib().th2d_set_cg_resident(ctx.ptr, 1)
    for (x1, i1), (x0, i0), b in zip(out[1], out[0], rhs):
        for u, v, p, q in zip(x1, x0, i1, i0):
            assert p.iterations == q.iterations and np.array_equal(u, v)
        _check(oracle, [(L, A, bb) for (L, A, _), bb in zip(rest, b)], x1, i1, 1e-10)


@pytest.mark.parametrize("dims", [[(128, 128)] * 4, [(96, 96), (70, 66)]])
def test_fp64_timeout_falls_back(hmc, oracle, N, dims):
    """A wait of the FP64 resident kernel that gives up (a limit of 0 polls,
    every workgroup still exits): the step kernel solves the batch."""
    batch, rest = _batch(hmc, oracle, dims)
    ctx, bs = batch.ctx, [b for _, _, b in rest]
    p = hmc.cg_params(tol_rel=1e-12)
    n0 = _fallbacks(N, ctx)
    N.check(N.lib().th2d_set_cg_spin_limit(ctx.ptr, 0), "spin")
    try:
        xs, infos = batch.fmdm_invert_cg(bs, p)
        assert _kernel(N, ctx) == STEP and _fallbacks(N, ctx) > n0
    finally:
        N.check(N.lib().th2d_set_cg_spin_limit(ctx.ptr, -1), "spin")
    _check(oracle, rest, xs, infos, 1e-12)
    batch.fmdm_invert_cg(bs, p)
    assert _kernel(N, ctx) == RESIDENT


@pytest.mark.parametrize("dims, mu, anti", [
    ([(16, 16), (8, 12)], 0.0, (1, 1)),      # 256 threads, one site each
    ([(16, 32), (6, 10)], 0.0, (1, 1)),      # two
    ([(24, 40), (32, 32)], 0.0, (1, 1)),     # four
    ([(32, 64), (34, 60)], 0.0, (1, 1)),     # 1024 threads, two
    ([(16, 16), (12, 20)], 0.1, (1, 1)),     # e^{+-mu} factors, the stochastic force
    ([(34, 60)], 0.1, (1, 0)),
    ([(16, 32)], 0.0, (0, 1)),
])
def test_fused_md_steps_match_the_general_ones(hmc, N, dims, mu, anti):
    """One trajectory with the MD steps fused (k_md_small) and by the general
    operations (th2d_set_cg_small off).  Both solve to 1e-12; the links differ
    by what the solves leave open, about nsteps h F kappa tol <= 8 x 0.05 x 10
    x 400 x 1e-12 = 2e-9, and the actions (of order V) by that times sqrt(V)."""
    ctx = hmc.Context.get()
    out = {}
    try:
        for on in (1, 0):
            N.check(N.lib().th2d_set_cg_small(ctx.ptr, on), "small")
            lats = []
            for k, (nt, nx) in enumerate(dims):
                lat = hmc.StaggeredLattice(nt, nx, m=0.2, g=0.6, mu=mu, anti_t=anti[0],
                                           anti_x=anti[1])
                lat.random_links(90 + k)
                lats.append(lat)
            batch = hmc.ChainBatch(lats)
            res = batch.update_gauge(nsteps=8, traj_len=0.4, params=hmc.cg_params(tol_rel=1e-12),
                                     seed=11, counters=[3] * len(dims), u_accept=[0.0] * len(dims))
            assert _kernel(N, ctx) == (SMALL if on else STEP)
            out[on] = (res, [l.get_links() for l in lats])
    finally:
        N.lib().th2d_set_cg_small(ctx.ptr, 1)
    for (nt, nx), r1, r0, a1, a0 in zip(dims, out[1][0], out[0][0], out[1][1], out[0][1]):
        assert r1.status == 0 and r0.status == 0 and r1.cg_solves == r0.cg_solves
        assert r1.accepted == r0.accepted == 1
        assert np.max(np.abs(a1 - a0)) <= 2e-9
        assert np.max(np.abs(np.array(r1.acts) - np.array(r0.acts))) <= 2e-9 * np.sqrt(nt * nx)
        assert abs(r1.cg_iterations - r0.cg_iterations) <= max(4, r0.cg_iterations // 50)


@pytest.mark.parametrize("dims, kernel", [
    ([(512, 512), (64, 64), (96, 96)], BOTH),
    ([(64, 64)] + [(384, 384)] + [(128, 128)] * 7, BOTH),
    ([(384, 384), (96, 96)], STEP),          # the split would cost more than it saves
    ([(16, 16), (384, 384)], STEP),
])
@pytest.mark.parametrize("prec", [0, 2])
def test_split_batches(hmc, oracle, N, dims, kernel, prec):
    """Lattices larger than an XCD's resident workgroups beside smaller ones."""
    batch, rest = _batch(hmc, oracle, dims)
    tol = 1e-12 if prec == 0 else 1e-10
    xs, infos = batch.fmdm_invert_cg([b for _, _, b in rest],
                                     hmc.cg_params(tol_rel=tol, precision=prec))
    assert _kernel(N, batch.ctx) == kernel
    _check(oracle, rest, xs, infos, tol)
