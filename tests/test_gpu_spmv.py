"""K4 (SpMV / multi-field SpMM) and K3 (CSR -> CSC) on the GPU against the
oracle and scipy."""
import numpy as np
import pytest
import scipy.sparse as sp

from rbffd_amd.nodes import jittered_grid

pytestmark = pytest.mark.gpu


def _operator(ctx, X, n=31, p=7, polydeg=4):
    import rbffd_amd

    eng = rbffd_amd.Engine(ctx)
    Xd = ctx.to_device(X)
    col, vals, _ = eng.generate(Xd, Xd, p, n, polydeg, ["Lap", "Dx"])
    return eng, Xd, col, vals


@pytest.mark.parametrize("F", [1, 2, 4, 8])
@pytest.mark.parametrize("vtype", ["f64", "f32"])
def test_spmv_matches_oracle(ctx, O, F, vtype):
    X = jittered_grid(80, 70, 0.25, seed=6)
    N, n = len(X), 31
    print(f"spmv F={F} {vtype}", flush=True)
    eng, Xd, col, vals = _operator(ctx, X)
    rng = np.random.default_rng(F)
    x = rng.standard_normal((N, F)) if F > 1 else rng.standard_normal(N)
    xd = ctx.to_device(x)
    yd = ctx.empty(x.shape, np.float64)
    v = vals[0].get()
    if vtype == "f32":
        v = v.astype(np.float32)
    vd = ctx.to_device(v)
    eng.spmv(col, vd, xd, yd, uniform_n=n)
    y = yd.get()
    rowptr = np.arange(N + 1, dtype=np.int64) * n
    ref = O.spmv_csr(rowptr, col.get().ravel(), v.astype(np.float64).ravel(), x)
    scale = np.abs(v).max() * np.abs(x).max() * n
    assert np.abs(y - ref).max() <= 1e-13 * scale
    # explicit rowptr path, alpha/beta
    rpd = ctx.to_device(rowptr)
    y2 = ctx.to_device(np.ones_like(x))
    eng.spmv(col, vd, xd, y2, rowptr=rpd, alpha=2.0, beta=-1.0)
    assert np.abs(y2.get() - (2 * ref - 1)).max() <= 2e-13 * scale
    # a locality order changes which rows run together, not the results
    order = eng.locality_order(Xd)
    oh = order.get()
    assert np.array_equal(np.sort(oh), np.arange(N))
    y3 = ctx.empty(x.shape, np.float64)
    eng.spmv(col, vd, xd, y3, uniform_n=n, order=order)
    assert np.array_equal(y3.get(), y)


@pytest.mark.parametrize("M", [1, 15, 17, 70])
@pytest.mark.parametrize("vtype", ["f64", "f32"])
@pytest.mark.parametrize("lens", ["ragged", 1, 4, 31, 32, 33, 64, 67])
def test_eight_fields_row_lengths(ctx, M, vtype, lens):
    # rows of every length around the 4 entries of a step and the 32 of a pass,
    # in plain products and plans; node 0, which padded entries read,
    # holds a NaN and is no row's column.  An entry's product is rounded once in
    # its sum, and sums of at most 70 terms lie within 70 ulps of sum |v x|.
    import rbffd_amd

    print(f"8 fields M={M} {vtype} lens={lens}", flush=True)
    rng = np.random.default_rng(M)
    N = 200
    n = np.resize([0, 1, 3, 4, 5, 31, 32, 33, 36, 63, 64, 65, 70], M) if lens == "ragged" else np.full(M, lens)
    rowptr = np.concatenate([[0], np.cumsum(n)]).astype(np.int64)
    col = rng.integers(1, N, rowptr[-1]).astype(np.int32)
    v = rng.standard_normal(rowptr[-1]).astype(np.float32 if vtype == "f32" else np.float64)
    x = rng.standard_normal((N, 8))
    # copied: abs() sums duplicates in place
    A = sp.csr_matrix((v.astype(np.float64), col, rowptr), shape=(M, N), copy=True)
    ref, mag = A @ np.where(np.arange(N)[:, None] == 0, 0.0, x), abs(A) @ abs(x)
    x[0] = np.nan
    eng = rbffd_amd.Engine(ctx)
    how = dict(rowptr=ctx.to_device(rowptr)) if lens == "ragged" else dict(uniform_n=int(lens))
    cd, vd, xd = ctx.to_device(col), ctx.to_device(v), ctx.to_device(x)
    order = ctx.to_device(rng.permutation(M).astype(np.int32))
    y = [ctx.empty((M, 8), np.float64) for _ in range(3)]
    eng.spmv(cd, vd, xd, y[0], **how)
    eng.spmv(cd, vd, xd, y[1], order=order, **how)
    plan = eng.spmv_plan(cd, vd, M, N, order=order, **how)
    plan.apply(xd, y[2])
    out = [a.get() for a in y]
    plan.close()
    assert (np.abs(out[0] - ref) <= 70 * 2.0**-52 * mag).all()
    assert np.array_equal(out[1], out[0]) and np.array_equal(out[2], out[0])


def test_csr_to_csc_matches_sparse(ctx, O):
    X = jittered_grid(60, 50, 0.25, seed=7)
    N, n = len(X), 31
    print("csr -> csc", flush=True)
    eng, Xd, col, vals = _operator(ctx, X)
    cp, rv, cv, used = eng.csr_to_csc(col, vals, N, index_base=0)
    c = col.get()
    rows = np.repeat(np.arange(N), n)
    for o in range(2):
        rcp, rrv, rnz, shape = O.sparse_csc(rows, c.ravel(), vals[o].get().ravel())
        assert used == shape[1]
        assert np.array_equal(cp.get()[: used + 1], rcp)
        assert np.array_equal(rv.get(), rrv)
        assert np.array_equal(cv[o].get(), rnz)
    cp1, rv1, _, _ = eng.csr_to_csc(col, vals[:1], N, index_base=1)
    assert np.array_equal(cp1.get(), cp.get() + 1)
    assert np.array_equal(rv1.get(), rv.get() + 1)
