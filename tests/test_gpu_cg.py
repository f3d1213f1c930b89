"""The PCG's dots: formed in the row sums of the apply or by a launch of their
own, the bits of a column depend on its rows alone and not on the columns beside
it, on profiling or on the path of the apply."""
import ctypes as C

import numpy as np
import pytest

import dfx
import oracle as O
from gpu_helpers import Ops
from problems import c1_like, enriched, guess, hanging

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52
# every lane count of the row sums with p.w (up to 8, 16, 32, 64, 128 columns, even)
# and of the separate dots (up to 8, 16, 32, more), odd counts, more than 128
WIDTHS = (1, 2, 3, 6, 8, 9, 12, 16, 20, 33, 40, 66, 100, 128, 130)


def mv(ctx, a, dtype=dfx.F64):
    return dfx.MultiVector.from_numpy(ctx, a, dtype)


@pytest.fixture(scope="module")
def probs():
    return {"c1": c1_like(n=3), "hang3": hanging(p=3), "enr": enriched(p=2, n=4)}


def jacobi(P, key="K"):
    d = P.arrays()
    diag, off, moff = np.zeros(P.nDofs), 0, 0
    for n in d["cellNdofs"]:
        ids = d["cellMap"][off:off + n]
        diag[ids] += np.diag(d[key][moff:moff + n * n].reshape(n, n, order="F"))
        off += n
        moff += n * n
    diag = P.c2p(diag.reshape(-1, 1))[:, 0]
    diag[d["rows"]] = 1.0
    return 1.0 / diag


@pytest.mark.parametrize("name", ["c1", "hang3"])
@pytest.mark.parametrize("B", WIDTHS)
def test_first_step_length_is_the_quotient_of_the_dots(ctx, probs, name, B):
    """One iteration from zero gives x = (z.r / p.w) p with r = b, p = z = d o b and
    w = K p (the apply leaves p with its constrained rows set from their parents);
    every column has converged then for this tolerance."""
    P = probs[name]
    ops = Ops(ctx, P)
    dinv = jacobi(P)
    b = P.c2p(guess(P, B, seed=B))
    x = dfx.MultiVector(ctx, P.nDofs, B)
    cg = dfx.CGLinearSolver(ctx, 1, 0.0, 0.9, 1e10)
    assert cg.solve(ops.K, dfx.DiagonalOperator(ctx, dinv), mv(ctx, b), x) == 0
    p = P.p2c(dinv[:, None] * b)
    w = P.apply(O.OP_K, p.copy())
    want = ((p * b).sum(axis=0) / (p * w).sum(axis=0)) * p
    # N-long sums of terms whose absolute sum is below twice the sum here, and
    # the apply's sums of up to 64 products from up to 8 cells
    tol = 2 * EPS * (2 * P.nDofs + 512)
    assert np.abs(x.to_numpy() - want).max() <= tol * np.abs(want).max()


@pytest.mark.parametrize("name", ["c1", "hang3", "enr"])
def test_a_column_does_not_depend_on_its_neighbours(ctx, probs, name, monkeypatch):
    """The solution of a right-hand side is the same bits alone, in any batch, while
    the operator is profiled and where the apply's slots are refused; the residual
    is below the tolerance and the iterations are the oracle's."""
    P = probs[name]
    ops = Ops(ctx, P)
    dinv = jacobi(P)
    pc = dfx.DiagonalOperator(ctx, dinv)
    n = max(WIDTHS)
    b = P.c2p(guess(P, n, seed=6))

    def solve(B, K):
        x = dfx.MultiVector(ctx, P.nDofs, B)
        cg = dfx.CGLinearSolver(ctx, 2000, 1e-12, 1e-10, 1e10)
        assert cg.solve(K, pc, mv(ctx, np.ascontiguousarray(b[:, :B])), x) == 0
        return x.to_numpy(), cg.iterations

    want, iters = solve(n, ops.K)
    rc, _, ito = P.cg(O.OP_K, dinv, b, abs_tol=1e-12, rel_tol=1e-10)
    assert rc == 0 and abs(iters - ito) <= 1
    res = b - P.apply(O.OP_K, want.copy())
    # the recurrence's residual against the true one: rounding of each update
    bound = 1e-10 * np.linalg.norm(b, axis=0).max() + \
        10 * ito * EPS * np.abs(want).max() * np.abs(P.arrays()["K"]).max() * np.sqrt(P.nDofs)
    assert np.linalg.norm(res, axis=0).max() <= bound
    rows = int(P.arrays()["cellNdofs"].sum())
    for B in WIDTHS:
        assert np.array_equal(solve(B, ops.K)[0], want[:, :B]), B
        if B not in (1, 8, 12, 33, 128):
            continue
        ops.K.set_profiling(True)
        assert np.array_equal(solve(B, ops.K)[0], want[:, :B]), B
        ops.K.set_profiling(False)
        fresh = Ops(ctx, P).K                      # no slots yet, work space allocated
        monkeypatch.setenv("DFX_MAX_ALLOC_BYTES", str(rows * B * 8 - 1))
        got = solve(B, fresh)[0]
        monkeypatch.delenv("DFX_MAX_ALLOC_BYTES")
        assert np.array_equal(got, want[:, :B]), B


@pytest.mark.parametrize("dtype", [dfx.F64, dfx.F32])
@pytest.mark.parametrize("N", [1, 63, 64, 65, 1000, 70001])
def test_dots_of_a_column_in_any_batch(ctx, N, dtype):
    """Blocks of 64 rows and more, cut-off lanes and every thread shape."""
    npd = np.float64 if dtype == dfx.F64 else np.float32
    n = 66
    X, Y = (O.rng_uniform(s, -1, 1, N * n).reshape(N, n).astype(npd) for s in (3, 4))
    want = None
    for B in (66, 1, 8, 9, 16, 17, 32, 33):
        got = np.array(mv(ctx, np.ascontiguousarray(X[:, :B]), dtype).dots(
            mv(ctx, np.ascontiguousarray(Y[:, :B]), dtype)))
        if want is None:
            want = got
            ref = (X.astype(np.float64) * Y).sum(axis=0)
            bound = EPS * (N + 2) * np.abs(X.astype(np.float64) * Y).sum(axis=0)
            assert (np.abs(got - ref) <= bound).all()
        assert np.array_equal(got, want[:B]), B


def test_work_space_of_a_solve():
    """r, w, z, p and two copies of x: the pipelined fused solve holds six arrays."""
    own = dfx.Context(0)
    N, B = 1 << 20, 8
    one = dfx.DiagonalOperator(own, np.ones(N))
    b, x = dfx.MultiVector(own, N, B), dfx.MultiVector(own, N, B)
    b.fill_random(1, -1.0, 1.0)
    one.apply(b, x)                      # the kernels are loaded
    x.set(0.0)

    def free():
        own.synchronize()
        f, t = C.c_size_t(), C.c_size_t()
        assert dfx._lib.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    before = free()
    assert dfx.CGLinearSolver(own, 10, 1e-12, 1e-10, 1e10).solve(one, one, b, x) == 0
    arrays = (before - free()) / (8.0 * N * B)
    assert 6.0 <= arrays < 6.5
    own.close()
