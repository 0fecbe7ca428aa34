"""The triangular solves of the blocked LU (U12 = L11^-1 A12) and of its
inverse are substitutions: where a 32 x 32 diagonal block is ill-conditioned
(unit triangular with about -7/8 off the diagonal, inverse entries up to
1.9^30) and the solution is of the order of 1, the residual stays within the
bound of substitution.  Substitution and the updates before it form every
element from at most n products, so |b - T x| <= gamma |T| |x| with
gamma = (n + 2) u to first order, u half the type's spacing; the bound is
twice that, for the partial sums of the updates."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N1 = 128  # a block of the factorisation


@pytest.fixture(scope="module")
def bag():
    from thirring2d_amd import bag as B
    return B


@pytest.fixture(scope="module")
def native():
    from thirring2d_amd import _native as N
    return N


def _steep(n, lower):
    """Unit triangular, 64ths in [-1, -3/4] off the diagonal of its 32 x 32
    diagonal blocks (all of -1 would let the products round as substitution
    does, every row twice the one before)."""
    r = np.random.default_rng(n)
    T = np.eye(n)
    for k in range(0, n, 32):
        e = min(k + 32, n)
        T[k:e, k:e] -= np.tril(r.integers(48, 65, size=(e - k, e - k)) / 64, -1)
    return T if lower else T.T.copy()


@pytest.fixture(params=["f64", "f32"])
def prec(request, native):
    return ((native.PREC_F64, np.float64) if request.param == "f64"
            else (native.PREC_F32, np.float32))


@pytest.fixture(params=[1, 0])
def mfma(request, native):
    native.lib().th2d_set_dense_mfma(request.param)
    yield request.param
    native.lib().th2d_set_dense_mfma(1)


@pytest.mark.parametrize("cols", [64, 1, 37, 200])
def test_u12_by_substitution(bag, prec, mfma, cols):
    p, dt = prec
    r = np.random.default_rng(3 + cols)
    L = _steep(N1, True)
    A = np.zeros((N1 + cols, N1 + cols))
    A[:N1, :N1] = L
    A[:N1, N1:] = L @ r.normal(size=(N1, cols))
    A[N1:, N1:] = np.eye(cols)
    A = A.astype(dt)
    db = bag.DenseBatch([A], p).lu()
    F = db.matrices()[0].astype(np.longdouble)
    assert np.array_equal(db.piv.download((N1 + cols,), np.int32), np.arange(N1 + cols))
    assert np.array_equal(np.tril(F[:N1, :N1], -1) + np.eye(N1), L)
    U12 = F[:N1, N1:]
    res = np.abs(A[:N1, N1:].astype(np.longdouble) - L.astype(np.longdouble) @ U12)
    gamma = 2 * (N1 + 2) * np.finfo(dt).eps / 2
    assert np.all(res <= gamma * (np.abs(L) @ np.abs(U12)))


@pytest.mark.parametrize("n2", [64, 1, 37, 200])
@pytest.mark.parametrize("lower", [True, False])
def test_inverse_by_substitution(bag, prec, mfma, lower, n2):
    """A = L with L22^-1 L21 of the order of 1/64 (U = 1), and A = U with
    U11^-1 U12 of that order (L = 1)."""
    p, dt = prec
    r = np.random.default_rng(5 + n2)
    if lower:  # the steep block below, its triangles on the solve's slices
        n1, m2 = (n2 + 31) // 32 * 32, N1
        T22 = _steep(m2, True)
        A = np.eye(n1 + m2)
        A[n1:, n1:] = T22
        A[n1:, :n2] = -T22 @ (r.uniform(-1, 1, size=(m2, n2)) / 64)
    else:
        T11 = _steep(N1, False)
        A = np.eye(N1 + n2)
        A[:N1, :N1] = T11
        A[:N1, N1:] = -T11 @ (r.uniform(-1, 1, size=(N1, n2)) / 64)
    A = A.astype(dt)
    n = A.shape[0]
    db = bag.DenseBatch([A], p).lu()
    assert np.array_equal(db.matrices()[0], A)
    X = db.inverse()[0].astype(np.longdouble)
    T = A.astype(np.longdouble)
    res = np.abs(T @ X - np.eye(n))
    gamma = 2 * (n + 2) * np.finfo(dt).eps / 2
    assert np.all(res <= gamma * (np.abs(T) @ np.abs(X)))
