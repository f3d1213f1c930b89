"""The slot path of the cell-wise apply (every cell's product to its map
slots, then row sums) against the colour-by-colour path, which
dfx_op_apply_noalloc takes at any size: bit for bit, over column counts at the
edges of the column tiles and 16-byte vectors, both precisions, constraints
with and without parents, enriched rows and every size class."""
import ctypes as C

import numpy as np
import pytest

import dfx
import oracle as O
from gpu_helpers import Ops
from problems import c1_like, enriched, guess, hanging

pytestmark = pytest.mark.gpu


def mv(ctx, a, dtype=dfx.F64):
    return dfx.MultiVector.from_numpy(ctx, a, dtype)


@pytest.fixture(scope="module")
def probs():
    atoms = [(-1.0, 0.5, 0.2, 1), (1.2, -0.8, 0.6, 6), (0.3, 1.4, -1.1, 8)]
    return {"c1": c1_like(n=3), "hang3": hanging(p=3), "enr": enriched(p=2, n=4),
            "wide": O.Problem.build(p=4, n=(3, 3, 3), lo=(-12.,) * 3, hi=(12.,) * 3, atoms=atoms,
                                    enrich=True, nq_enr=6)}


@pytest.mark.parametrize("name", ["c1", "hang3", "enr", "wide"])
@pytest.mark.parametrize("dtype", [dfx.F64, dfx.F32])
def test_slot_apply_equals_colour_apply(ctx, probs, name, dtype):
    P = probs[name]
    ops = Ops(ctx, P)
    npd = np.float64 if dtype == dfx.F64 else np.float32
    for B in (1, 2, 3, 5, 16, 17, 31, 33, 40, 48, 49, 64, 66, 72, 80, 81, 101, 130):
        X = O.rng_uniform(B, -1, 1, P.nDofs * B).reshape(P.nDofs, B).astype(npd)
        Xa, Xb = mv(ctx, X, dtype), mv(ctx, X, dtype)
        Ya, Yb = (dfx.MultiVector(ctx, P.nDofs, B, dtype) for _ in range(2))
        ops.H.apply(Xa, Ya)
        ops.H.apply_noalloc(Xb, Yb)
        assert np.array_equal(Ya.to_numpy(), Yb.to_numpy()), (name, B)
        assert np.array_equal(Xa.to_numpy(), Xb.to_numpy()), (name, B)   # the same P2C on X


@pytest.mark.parametrize("name", ["c1", "hang3", "wide"])
@pytest.mark.parametrize("dtype", [dfx.F64, dfx.F32])
def test_folded_inverse_equals_the_two_applies_at_any_width(ctx, probs, name, dtype):
    """M^-1 folded into the gather against M^-1's apply then H's colour path
    (X gets the same parent->child update)."""
    P = probs[name]
    ops = Ops(ctx, P)
    npd = np.float64 if dtype == dfx.F64 else np.float32
    for B in (1, 3, 13, 40, 72):
        X = O.rng_uniform(B, -1, 1, P.nDofs * B).reshape(P.nDofs, B).astype(npd)
        Xa, Xb = mv(ctx, X, dtype), mv(ctx, X, dtype)
        Ya, Yb, Z = (dfx.MultiVector(ctx, P.nDofs, B, dtype) for _ in range(3))
        ops.H.apply_after_inverse(ops.Minv, Xa, Ya)
        ops.Minv.apply(Xb, Z)
        ops.H.apply_noalloc(Z, Yb)
        assert np.array_equal(Ya.to_numpy(), Yb.to_numpy()), (name, B)
        assert np.array_equal(Xa.to_numpy(), Xb.to_numpy()), (name, B)


@pytest.mark.parametrize("B", [3, 13, 40])
@pytest.mark.parametrize("prec", [dfx.PREC_FP64, dfx.PREC_MIXED])
def test_residual_step_in_the_row_sums_is_bit_identical(ctx, probs, B, prec, monkeypatch):
    P = probs["wide"]
    ops = Ops(ctx, P)
    X = guess(P, B, seed=B)
    lo, hi, beta = P.lanczos(O.rng_uniform(2, -1, 1, P.nDofs))
    a, c = lo, hi + beta / 10
    b = a + 0.05 * (c - a)
    outs = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("DFX_FUSE_RES", fuse)
        G, V = mv(ctx, X), dfx.MultiVector(ctx, P.nDofs, B)
        s = dfx.ChebyshevFilteredEigenSolver(ctx, a, b, c, 7, 1e-14, G, True, 0, prec)
        eig = np.linspace(a, b, B)
        assert s.solve(ops.H, eig, V, True, ops.M, ops.Minv) == 0
        outs.append((eig, V.to_numpy()))
    assert np.array_equal(outs[0][0], outs[1][0]) and np.array_equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("dtype", [dfx.F64, dfx.F32])
@pytest.mark.parametrize("B", [4, 5])
def test_addresses_of_one_value_alignment(ctx, probs, dtype, B):
    """Caller-owned memory that starts one value past a 16-byte boundary."""
    P = probs["enr"]
    ops = Ops(ctx, P)
    npd = np.float64 if dtype == dfx.F64 else np.float32
    X = O.rng_uniform(B, -1, 1, P.nDofs * B).reshape(P.nDofs, B).astype(npd)
    want = dfx.MultiVector(ctx, P.nDofs, B, dtype)
    ops.H.apply(mv(ctx, X, dtype), want)

    def shifted():
        own = dfx.MultiVector(ctx, P.nDofs * B + 8, 1, dtype)
        m = dfx.MultiVector.__new__(dfx.MultiVector)
        m.ctx, m.N, m.B, m.dtype, m.h, m.own = ctx, P.nDofs, B, dtype, C.c_void_p(), own
        ctx.check(dfx._lib.dfx_mv_wrap(ctx.h, own.device_ptr + np.dtype(npd).itemsize, P.nDofs, B,
                                       dtype, C.byref(m.h)))
        return m

    Xs, Ys = shifted(), shifted()
    Xs.upload(X)
    ops.H.apply(Xs, Ys)
    assert np.array_equal(Ys.to_numpy(), want.to_numpy())


@pytest.mark.parametrize("cells", [30, 31, 40])
def test_rows_of_many_cells_and_of_none(ctx, cells):
    """Cells that all share one dof (a row of up to 30 cells has slot lists,
    more fall back to one launch per colour) and a dof in no cell."""
    n = cells + 2                                   # dof cells + 1: in no cell
    cmap = np.stack([np.zeros(cells, int), np.arange(1, cells + 1)], axis=1)
    A = O.rng_uniform(cells, -1, 1, cells * 4).reshape(cells, 2, 2)
    op = dfx.CellOperator(ctx, np.full(cells, 2), cmap.ravel(), A.ravel(), n)
    X = O.rng_uniform(3, -1, 1, n * 6).reshape(n, 6)
    Y = dfx.MultiVector(ctx, n, 6)
    Y.set(7.0)
    op.apply(mv(ctx, X), Y)
    ref = np.zeros_like(X)
    for e in range(cells):
        # y_cell = x_cell A (column-major blocks, both stored row by row here)
        ref[cmap[e]] += A[e] @ X[cmap[e]]
    # sums of at most `cells` + 2 products per entry
    assert np.abs(Y.to_numpy() - ref).max() <= (cells + 2) * 2.0 ** -52 * cells


@pytest.mark.parametrize("dtype", [dfx.F64, dfx.F32])
def test_cells_with_the_same_matrix_share_it(ctx, probs, dtype):
    """Cells of bitwise equal matrices share one stored copy; one that differs in
    a single bit does not, and update_cells may turn either into the other;
    against numpy's cell-by-cell sums and a freshly made operator."""
    P = probs["c1"]
    d = P.arrays()
    ops = Ops(ctx, P)
    n = int(d["cellNdofs"][0])
    nc = len(d["cellNdofs"])
    K0 = d["K"][:n * n]
    uniform = np.tile(K0, nc)
    one_bit = uniform.copy()
    one_bit[n * n * (nc // 2) + 5] = np.nextafter(one_bit[n * n * (nc // 2) + 5], 10.0)
    distinct = (uniform.reshape(nc, -1) * (1.0 + np.arange(nc)[:, None] / 64.0)).ravel()
    npd = np.float64 if dtype == dfx.F64 else np.float32
    X = guess(P, 10, seed=4).astype(npd)
    off = np.concatenate([[0], np.cumsum(d["cellNdofs"])]).astype(int)
    cons_rows = d["rows"]

    def reference(mats):
        Z, Y = X.astype(np.float64), np.zeros((P.nDofs, 10))
        Z[cons_rows] = 0
        for e in range(nc):
            i = d["cellMap"][off[e]:off[e + 1]].astype(int)
            np.add.at(Y, i, mats[e * n * n:(e + 1) * n * n].reshape(n, n) @ Z[i])
        Y[cons_rows] = 0
        return Y

    def result(op):
        Y = dfx.MultiVector(ctx, P.nDofs, 10, dtype)
        op.apply(mv(ctx, X, dtype), Y)
        Yc = dfx.MultiVector(ctx, P.nDofs, 10, dtype)
        op.apply_noalloc(mv(ctx, X, dtype), Yc)
        assert np.array_equal(Y.to_numpy(), Yc.to_numpy())
        return Y.to_numpy()

    def make(mats):
        return dfx.CellOperator(ctx, d["cellNdofs"], d["cellMap"], mats, P.nDofs, P.nClassical,
                                ops.cons, keep_fp32=True)

    unit = make(uniform).info()["matBytesF64"]
    assert make(one_bit).info()["matBytesF64"] == 2 * unit
    assert make(distinct).info()["matBytesF64"] == nc * unit
    op = make(uniform)
    # n-term products and up to 8 cells added per row, each rounded in `dtype`
    eps = np.finfo(npd).eps
    for mats in (uniform, distinct, one_bit, uniform):
        op.update_cells(mats)
        got, ref = result(op), reference(mats)
        assert np.abs(got - ref).max() <= (n + 10) * eps * np.abs(mats).max() * n
        assert np.array_equal(got, result(make(mats)))


@pytest.mark.parametrize("dtype", [dfx.F64, dfx.F32])
def test_profiled_bytes_count_a_shared_matrix_once(ctx, probs, dtype, monkeypatch):
    """The bytes of a profile hold every distinct matrix of a launch once, on the
    slot path (one launch here) and colour by colour (where the slots are refused);
    the flops those of every cell; an update changes the bytes with the matrices."""
    P = probs["c1"]
    d = P.arrays()
    n, nc, B = int(d["cellNdofs"][0]), len(d["cellNdofs"]), 8
    size = 8 if dtype == dfx.F64 else 4
    uniform = np.tile(d["K"][:n * n], nc)
    distinct = (uniform.reshape(nc, -1) * (1.0 + np.arange(nc)[:, None] / 64.0)).ravel()
    X, Y = (dfx.MultiVector(ctx, P.nDofs, B, dtype) for _ in range(2))
    for limit in (None, int(d["cellNdofs"].sum()) * B * size - 1):
        op = dfx.CellOperator(ctx, d["cellNdofs"], d["cellMap"], uniform, P.nDofs,
                              P.nClassical, Ops(ctx, P).cons, keep_fp32=True)
        got = []
        for mats in (None, distinct):
            if mats is not None:
                op.update_cells(mats)
            if limit:
                monkeypatch.setenv("DFX_MAX_ALLOC_BYTES", str(limit))
            op.set_profiling(True)
            op.apply(X, Y)
            got.append(op.profile(reset=True))
            monkeypatch.delenv("DFX_MAX_ALLOC_BYTES", raising=False)
        launches = op.info()["nColors"] if limit else 1
        assert [g["launches"] for g in got] == [launches, launches]
        assert got[0]["flops"] == got[1]["flops"] == 2.0 * B * nc * n * n
        assert got[1]["bytes"] - got[0]["bytes"] == size * (nc - launches) * n * n


def test_a_refused_update_leaves_the_operator_as_it_was(ctx, monkeypatch):
    """Where an update from equal to distinct cell matrices is refused for want of
    memory the operator keeps its matrices (FP64, FP32 and the colour-by-colour
    path); it needs no more than the copy of the caller's matrices."""
    P = c1_like(n=3, p=2)
    d = P.arrays()
    ops = Ops(ctx, P)
    n, nc = int(d["cellNdofs"][0]), len(d["cellNdofs"])
    uniform = np.tile(d["K"][:n * n], nc)
    distinct = (uniform.reshape(nc, -1) * (1.0 + np.arange(nc)[:, None] / 64.0)).ravel()

    def make(mats):
        return dfx.CellOperator(ctx, d["cellNdofs"], d["cellMap"], mats, P.nDofs, P.nClassical,
                                ops.cons, keep_fp32=True)

    def results(op):
        out = []
        for dtype, npd in ((dfx.F64, np.float64), (dfx.F32, np.float32)):
            X = guess(P, 6, seed=8).astype(npd)
            for call in (op.apply, op.apply_noalloc):
                Y = dfx.MultiVector(ctx, P.nDofs, 6, dtype)
                call(mv(ctx, X, dtype), Y)
                out.append(Y.to_numpy())
        return out

    op, fresh = make(uniform), make(distinct)
    before, info = results(op), op.info()
    assert fresh.info()["matBytesF64"] > distinct.nbytes
    monkeypatch.setenv("DFX_MAX_ALLOC_BYTES", str(distinct.nbytes - 1))
    with pytest.raises(dfx.DfxError, match="DFX_MAX_ALLOC_BYTES"):
        op.update_cells(distinct)
    assert op.info() == info
    for a, b in zip(results(op), before):
        assert np.array_equal(a, b)
    # room for the matrices as the caller holds them is enough
    monkeypatch.setenv("DFX_MAX_ALLOC_BYTES", str(distinct.nbytes))
    op.update_cells(distinct)
    monkeypatch.delenv("DFX_MAX_ALLOC_BYTES")
    for a, b in zip(results(op), results(fresh)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("call", ["apply", "apply_noalloc"])
def test_a_captured_apply_outlives_an_update(ctx, probs, call):
    """A caller's graph of an apply gives the new matrices' products after an update
    that changes how many of them differ."""
    P = probs["c1"]
    d = P.arrays()
    B, n, nc = 8, int(d["cellNdofs"][0]), len(d["cellNdofs"])
    uniform = np.tile(d["K"][:n * n], nc)
    distinct = (uniform.reshape(nc, -1) * (1.0 + np.arange(nc)[:, None] / 64.0)).ravel()
    ops = Ops(ctx, P)

    def make(mats):
        return dfx.CellOperator(ctx, d["cellNdofs"], d["cellMap"], mats, P.nDofs, P.nClassical,
                                ops.cons)

    op = make(uniform)
    X, Y = dfx.MultiVector(ctx, P.nDofs, B), dfx.MultiVector(ctx, P.nDofs, B)
    ops.H.apply_noalloc(X, Y)                        # the kernels are loaded
    ctx.synchronize()
    hip, stream, graph, run = dfx._lib, C.c_void_p(), C.c_void_p(), C.c_void_p()
    assert hip.dfx_ctx_stream(ctx.h, C.byref(stream)) == 0
    assert hip.hipStreamBeginCapture(stream, 0) == 0
    try:
        getattr(op, call)(X, Y)
    finally:
        assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
    for seed, mats in enumerate((uniform, distinct, uniform)):
        op.update_cells(mats)
        Xs, want = guess(P, B, seed=seed), dfx.MultiVector(ctx, P.nDofs, B)
        make(mats).apply(mv(ctx, Xs), want)
        X.upload(Xs)
        Y.set(0.0)
        assert hip.hipGraphLaunch(run, stream) == 0
        ctx.synchronize()
        assert np.array_equal(Y.to_numpy(), want.to_numpy())
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0


@pytest.mark.parametrize("name", ["c1", "hang3", "wide"])
@pytest.mark.parametrize("dtype", [dfx.F64, dfx.F32])
def test_applies_run_where_the_slots_cannot_be_had(ctx, probs, name, dtype, monkeypatch):
    """Operators whose slots are refused as out of memory apply colour by colour:
    plain, with M^-1 folded in, and tuned; the bits of the slot path."""
    P = probs[name]
    npd = np.float64 if dtype == dfx.F64 else np.float32
    size = np.dtype(npd).itemsize
    rows = int(P.arrays()["cellNdofs"].sum())
    for B in (8, 13, 40):
        X = O.rng_uniform(B, -1, 1, P.nDofs * B).reshape(P.nDofs, B).astype(npd)
        outs = []
        for limit in (None, rows * B * size - 1):
            ops = Ops(ctx, P)
            Xa, Xb = mv(ctx, X, dtype), mv(ctx, X, dtype)
            Ya, Yb, Yc = (dfx.MultiVector(ctx, P.nDofs, B, dtype) for _ in range(3))
            if limit:
                assert limit > P.nDofs * B * size        # vectors and work space are not
                monkeypatch.setenv("DFX_MAX_ALLOC_BYTES", str(limit))
            ops.H.apply(Xa, Ya)
            ops.H.apply_after_inverse(ops.Minv, Xb, Yb)
            ops.H.autotune(dtype, B, reps=1)
            ops.H.apply(Xa, Yc)
            monkeypatch.delenv("DFX_MAX_ALLOC_BYTES", raising=False)
            outs.append([v.to_numpy() for v in (Xa, Xb, Ya, Yb, Yc)])
        for a, b in zip(*outs):
            assert np.array_equal(a, b), (name, B)


@pytest.mark.parametrize("B", [8, 40, 72])
@pytest.mark.parametrize("prec", [dfx.PREC_FP64, dfx.PREC_MIXED])
def test_filter_runs_where_the_slots_cannot_be_had(ctx, probs, B, prec, monkeypatch):
    """The filter with the residual step in the colour kernel's scatter, eager
    and replayed, against the slot path: the same bits."""
    P = probs["wide"]
    lo, hi, beta = P.lanczos(O.rng_uniform(2, -1, 1, P.nDofs))
    a, c = lo, hi + beta / 10
    b = a + 0.05 * (c - a)
    X = guess(P, B, seed=B)
    size = 8 if prec == dfx.PREC_FP64 else 4
    limit = int(P.arrays()["cellNdofs"].sum()) * B * size - 1
    outs = []
    for graph in (False, True):
        G, V = mv(ctx, X), dfx.MultiVector(ctx, P.nDofs, B)
        s = dfx.ChebyshevFilteredEigenSolver(ctx, a, b, c, 7, 1e-14, G, True, 0, prec, graph)
        # with slots (this allocates the solver's work space), then fresh
        # operators that get none; the second of their passes replays the loop
        for ops, passes in ((Ops(ctx, P), 1), (Ops(ctx, P), 2)):
            for _ in range(passes):
                G.upload(X)
                eig = np.linspace(a, b, B)
                s.reinit(a, b, c, 7, 1e-14, G)
                assert s.solve(ops.H, eig, V, True, ops.M, ops.Minv) == 0
                outs.append((eig, V.to_numpy()))
                monkeypatch.setenv("DFX_MAX_ALLOC_BYTES", str(limit))
        monkeypatch.delenv("DFX_MAX_ALLOC_BYTES")
    for o in outs[1:]:
        assert np.array_equal(o[0], outs[0][0]) and np.array_equal(o[1], outs[0][1])


def test_a_captured_apply_outlives_the_slots(ctx, probs):
    """While a caller captures the stream an apply of a classical operator uses no
    slots: the first one allocates nothing, and a later one does not put the slots'
    address into the graph, which a wider apply moves.  Replays give the eager bits,
    with eager work between them."""
    P = probs["c1"]
    B = 8
    warm, ops = Ops(ctx, P), Ops(ctx, P)
    X, Y = dfx.MultiVector(ctx, P.nDofs, B), dfx.MultiVector(ctx, P.nDofs, B)
    warm.H.apply_noalloc(X, Y)                       # the kernels are loaded
    ctx.synchronize()
    hip, stream = dfx._lib, C.c_void_p()
    assert hip.dfx_ctx_stream(ctx.h, C.byref(stream)) == 0
    runs = []

    def capture():
        graph, run = C.c_void_p(), C.c_void_p()
        assert hip.hipStreamBeginCapture(stream, 0) == 0          # the strictest mode
        try:
            ops.H.apply(X, Y)
        finally:
            assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
        assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
        runs.append((graph, run))

    capture()
    for seed, wide in enumerate((8, 8, 16, 40)):
        Xw, want = guess(P, wide, seed=seed), dfx.MultiVector(ctx, P.nDofs, wide)
        ops.H.apply(mv(ctx, Xw), want)                            # eager: in slots
        if seed == 0:
            capture()
        X.upload(np.ascontiguousarray(Xw[:, :B]))
        for _, run in runs:
            Y.set(0.0)
            assert hip.hipGraphLaunch(run, stream) == 0
            ctx.synchronize()
            assert np.array_equal(Y.to_numpy(), want.to_numpy()[:, :B])
    for graph, run in runs:
        assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0


@pytest.mark.parametrize("dtype", [dfx.F64, dfx.F32])
@pytest.mark.parametrize("B", [33, 40, 48])
def test_widths_tuned_on_one_path_stay_there(ctx, probs, B, dtype, monkeypatch):
    """Three tiles of 16 columns is a width of the slot kernels only: tuned to it,
    an operator still applies colour by colour (without allocation, or where the
    slots are refused), with the bits of the untuned operator."""
    P = probs["wide"]
    npd = np.float64 if dtype == dfx.F64 else np.float32
    X = O.rng_uniform(B, -1, 1, P.nDofs * B).reshape(P.nDofs, B).astype(npd)
    ops = Ops(ctx, P)

    def run(call):
        Y = dfx.MultiVector(ctx, P.nDofs, B, dtype)
        call(mv(ctx, X, dtype), Y)
        return Y.to_numpy()

    before = run(ops.H.apply)
    monkeypatch.setenv("DFX_CELL_TUNE_NT", "3")
    assert set(ops.H.autotune(dtype, B, reps=1).values()) == {3}
    monkeypatch.delenv("DFX_CELL_TUNE_NT")
    assert np.array_equal(run(ops.H.apply), before)
    assert np.array_equal(run(ops.H.apply_noalloc), before)


def test_applies_on_both_sides_of_the_slot_limits(ctx):
    """1022 chained cells of 130 dofs: the widths next to the limits of the slot path
    (FP64 1 GiB of products; FP32 608 MiB above 128 columns where the colour path has
    its buffer kernel) take the path they should and give the same bits there."""
    cells, n = 1022, 130
    cmap = (120 * np.arange(cells)[:, None] + np.arange(n)).astype(np.uint32)
    N = int(cmap.max()) + 1
    A = O.rng_uniform(9, -1, 1, n * n)
    op = dfx.CellOperator(ctx, np.full(cells, n), cmap.ravel(), np.tile(A, cells), N,
                          keep_fp32=True)
    rows, colours = cells * n, op.info()["nColors"]
    assert colours > 1
    for dtype, size, limit, widths in ((dfx.F64, 8, 1024, (1010, 1012)),
                                       (dfx.F32, 4, 608, (1196, 1200, 1201))):
        for B in widths:
            slots = rows * B * size <= limit << 20 or B == 1201
            X, Ya, Yb = (dfx.MultiVector(ctx, N, B, dtype) for _ in range(3))
            X.fill_random(B, -1.0, 1.0)
            op.set_profiling(True)
            op.apply(X, Ya)
            assert op.profile(reset=True)["launches"] == (1 if slots else colours), B
            op.set_profiling(False)
            op.apply_noalloc(X, Yb)
            assert Ya.l2norms().min() > 0.0
            Ya.axpby(1.0, Ya, -1.0, Yb)
            assert not Ya.l2norms().any(), B
