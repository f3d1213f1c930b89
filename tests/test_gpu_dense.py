"""Gram matrices and subspace rotations at the edges of their column tiles
(1 to 257 columns: every kernel width, odd counts, the library path above 256)
and of their row chunks, through the Cholesky-Gram-Schmidt and Rayleigh-Ritz
entry points, against numpy."""
import numpy as np
import pytest

import dfx
import oracle as O

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


def diagonal(ctx, d):
    return dfx.DiagonalOperator(ctx, d)


@pytest.mark.parametrize("n", [1, 2, 3, 15, 16, 17, 32, 33, 63, 64, 65, 66, 101, 112, 113, 128, 129, 200,
                               208, 255, 256, 257])
def test_orthonormalization_and_ritz_at_every_width(ctx, n):
    for N in sorted({n, n + 1, 1031, 4099}):
        if N < n:
            continue
        rng = np.random.RandomState(n * 7 + N)
        # columns of a well-conditioned block: an orthonormal basis, slightly mixed
        X = np.linalg.qr(rng.uniform(-1, 1, (N, n)))[0]
        X = X + 0.3 * X @ np.triu(rng.uniform(-1, 1, (n, n)), 1) / max(1, n)
        m, h = rng.uniform(0.5, 2.0, N), rng.uniform(-1.0, 5.0, N)
        Xo = dfx.MultiVector(ctx, N, n)
        assert dfx.cholesky_gram_schmidt(ctx, dfx.MultiVector.from_numpy(ctx, X), Xo,
                                         diagonal(ctx, m)) == 0
        S = X.T @ (m[:, None] * X)
        L = np.linalg.cholesky(S)
        want = np.linalg.solve(L, X.T).T
        # backward errors of the N-long sums and of the factorization, amplified
        # by the factor's condition (below 10 here)
        tol = 10 * EPS * (n + np.sqrt(N)) * np.linalg.cond(L)
        got = Xo.to_numpy()
        assert np.abs(got - want).max() <= tol * max(1.0, np.abs(want).max()), (n, N)
        V = dfx.MultiVector(ctx, N, n)
        Y = np.linalg.qr(X)[0]
        rc, ev = dfx.rayleigh_ritz(ctx, diagonal(ctx, h), dfx.MultiVector.from_numpy(ctx, Y), V)
        assert rc == 0
        T = Y.T @ (h[:, None] * Y)
        tol = 10 * EPS * (n + np.sqrt(N)) * 6
        assert np.abs(ev - np.linalg.eigvalsh(T)).max() <= tol, (n, N)
        v = V.to_numpy()
        assert np.abs(v.T @ v - np.eye(n)).max() <= tol, (n, N)
        assert np.abs(v.T @ (h[:, None] * v) - np.diag(ev)).max() <= tol, (n, N)


def test_not_a_number_is_reported(ctx):
    """An odd count in one narrow tile gives finite results; a not-a-number value
    among its columns is reported as any failed factorization."""
    N, n = 300, 7
    X = O.rng_uniform(5, -1, 1, N * n).reshape(N, n)
    X = np.linalg.qr(X)[0]
    m = np.ones(N)
    Xo = dfx.MultiVector(ctx, N, n)
    assert dfx.cholesky_gram_schmidt(ctx, dfx.MultiVector.from_numpy(ctx, X), Xo,
                                     diagonal(ctx, m)) == 0
    assert np.isfinite(Xo.to_numpy()).all()
    X[4, 3] = np.nan
    rc = dfx.cholesky_gram_schmidt(ctx, dfx.MultiVector.from_numpy(ctx, X), Xo, diagonal(ctx, m))
    assert rc != 0


@pytest.mark.parametrize("n", [1, 15, 16, 17, 40, 200, 256, 257])
def test_rank_deficient_and_tiny_columns_are_reported(ctx, n):
    """A zero column, a column below the factor's 1e-14 limit and (from two
    columns on) equal unit vectors fail; a column of norm 1e-13 does not."""
    N = max(2 * n, 64)
    rng = np.random.RandomState(n)
    Q = np.linalg.qr(rng.uniform(-1, 1, (N, n)))[0]
    M, Xo = diagonal(ctx, np.ones(N)), dfx.MultiVector(ctx, N, n)

    def run(X):
        return dfx.cholesky_gram_schmidt(ctx, dfx.MultiVector.from_numpy(ctx, X), Xo, M)

    assert run(Q) == 0
    for j in sorted({0, n // 2, n - 1}):
        for scale, ok in ((0.0, False), (1e-15, False), (1e-13, True)):
            X = Q.copy()
            X[:, j] *= scale
            assert (run(X) == 0) == ok, (n, j, scale)
        if j:                                # equal columns whose pivot is exactly zero
            X = np.eye(N, n)
            assert run(X) == 0
            X[:, j] = X[:, 0]
            assert run(X) != 0
    assert run(Q) == 0                       # a failure leaves nothing behind
    assert np.abs(Xo.to_numpy() - Q).max() <= 50 * EPS * (n + np.sqrt(N))


@pytest.mark.parametrize("n", [2, 3, 17, 65, 100, 128, 150])
def test_projected_problems_with_nothing_to_reflect(ctx, n):
    """Diagonal and block-diagonal projected matrices (zero columns below the
    diagonal: reflectors of zero length), repeated values and a wide range of
    magnitudes: eigenvalues to the matrix norm, orthonormal vectors."""
    N = n + 5
    V = dfx.MultiVector(ctx, N, n)
    for h in (np.arange(N) * 1.0, np.ones(N), 10.0 ** np.linspace(-9, 3, N),
              np.where(np.arange(N) % 2, 1e-30, 2.0)):
        for X in (np.eye(N, n), np.eye(N, n)[:, ::-1].copy()):
            rc, ev = dfx.rayleigh_ritz(ctx, diagonal(ctx, h), dfx.MultiVector.from_numpy(ctx, X), V)
            assert rc == 0
            want = np.sort((X * (h[:, None] * X)).sum(axis=0))
            assert np.abs(ev - want).max() <= 20 * n * EPS * max(np.abs(want).max(), 1e-300)
            v = V.to_numpy()
            assert np.abs(v.T @ v - np.eye(n)).max() <= 20 * n * EPS
