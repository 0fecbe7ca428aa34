"""The inverse of batches of orders up to 32, or up to 64 with more matrices
than CUs (k_inv_small in csrc/dense.hip), beside the block solves, which the
same matrices reach in a batch with one of order 65."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
bag = pytest.importorskip("thirring2d_amd.bag")

ORDERS = [1, 2, 3, 4, 5, 15, 16, 17, 31, 32, 33, 61, 63, 64]


def _mats(seed, orders):
    r = np.random.default_rng(seed)
    return [r.normal(size=(n, n)) for n in orders]  # (pivots everywhere)


def _inverses(mats, prec):
    return bag.DenseBatch(mats, prec).lu().inverse()


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("orders", [ORDERS * 20, [3], [32], [33], [64], [1, 16, 31] * 3, [16] * 300])
def test_residual_and_block_path(prec, orders):
    """Both paths solve L Z = P and U X = Z by substitution, so that
    |P - L Z| <= gamma |L| |Z| and |Z - U X| <= gamma |U| |X|, gamma = (n + 2) u;
    |Z| <= |U| |X| to first order, and the factors' own error is gamma |L| |U|."""
    dt = np.float32 if prec else np.float64
    mats = [m.astype(dt) for m in _mats(len(orders), orders)]
    db = bag.DenseBatch(mats, prec).lu()
    X = db.inverse()
    F = db.matrices()
    Y = _inverses(mats + [np.eye(65)], prec)
    piv = np.split(db.piv.download((sum(orders),), np.int32), np.cumsum(orders)[:-1])
    for n, a, f, p, x, y in zip(orders, mats, F, piv, X, Y):
        L = np.tril(f.astype(np.longdouble), -1) + np.eye(n)
        U = np.triu(f.astype(np.longdouble))
        perm = np.arange(n)
        for j in range(n):
            perm[j], perm[p[j]] = perm[p[j]], perm[j]
        gamma = (n + 2) * np.finfo(dt).eps / 2
        for v in (x, y):
            v = v.astype(np.longdouble)
            res = np.abs(a.astype(np.longdouble)[perm] @ v - np.eye(n)[perm])
            assert np.all(res <= 3 * gamma * (np.abs(L) @ (np.abs(U) @ np.abs(v)))), n


def test_zero_pivot():
    """Below a zero pivot the columns of the inverse are finite, from it up
    they are not, in both paths alike."""
    a = np.triu(np.random.default_rng(2).uniform(0.5, 1.0, size=(24, 24)))
    a[13, 13] = 0.0
    (x,), (y, _) = _inverses([a], 0), _inverses([a, np.eye(65)], 0)
    assert np.array_equal(np.isfinite(x), np.isfinite(y))
    assert np.all(np.isfinite(x[14:])) and not np.any(np.isfinite(x[13, 13:]))


def test_refined_logdet_small_orders():
    """The FP64 correction from the small inverse (the columns not permuted):
    what is left of the FP32 error is its square, (n eps32)^2 times the
    condition (below 1e3 here: eps32^2 n^2 kappa^2 = 6e-5 at n = 64)."""
    r = np.random.default_rng(9)
    mats = [r.normal(size=(n, n)) + 4 * np.sqrt(n) * np.eye(n)[r.permutation(n)] for n in ORDERS * 20]
    d64 = bag.DenseBatch(mats, 0)
    la, sg = bag.DenseBatch(mats, 1).lu().logdet_refined(d64)
    for m, l, s in zip(mats, la, sg):
        s0, l0 = np.linalg.slogdet(m)
        kappa = np.linalg.cond(m)
        n = m.shape[0]
        assert s == s0
        assert abs(l - l0) <= (n * 2.0 ** -24 * kappa) ** 2 + n * kappa * 2.0 ** -52
