"""The null-space solve (odd PHS powers with polynomials of degree at least
(m - 1) / 2): weights against the high-precision oracle on node sets from
even to clustered, and what it hands to the pivoting kernel (duplicated and
nearly duplicated nodes, coordinates that are not finite) against that kernel
alone (RBFFD_NULLSPACE=0).

Bar: per-row relative error at most 1e-10, or 4 times that of an FP64 LU solve
of the same row's system, with the node set's median LU error as the least LU
error counted (single rows of an LU solve can be right by luck)."""
import numpy as np
import pytest

from rbffd_amd.nodes import jittered_grid

pytestmark = pytest.mark.gpu

# (PHS power, polynomial degree, stencil size)
SHAPES = [(3, 3, 20), (5, 3, 21), (7, 3, 21), (7, 4, 31), (9, 4, 31), (5, 5, 42), (7, 5, 43), (9, 6, 57)]
OPS = ["E", "Dx", "Dyy", "Dxy", "Lap", "Dxk", "Dyk"]


def _weights(ctx, X, st, p, polydeg, ops, k, method=1):
    import rbffd_amd

    eng = rbffd_amd.Engine(ctx)
    Xd = ctx.to_device(X)
    col, vals, status = eng.weights(Xd, Xd, ctx.to_device(st.astype(np.int32)), None, p, polydeg, ops, k=k,
                                    method=method)
    return col.get(), [v.get() for v in vals], status.get()


def _nodes(kind, seed):
    rng = np.random.default_rng(seed)
    if kind == "grid":
        return jittered_grid(23, 21, 0.3, seed=seed)  # 483 rows: three stencils past a full wavefront
    if kind == "uniform":
        return rng.uniform(0, 1, (401, 2))
    return np.concatenate([rng.uniform(0, 1, (200, 2)), 0.5 + 0.02 * rng.standard_normal((202, 2))])


@pytest.mark.parametrize("p,polydeg,n", SHAPES)
@pytest.mark.parametrize("kind", ["grid", "uniform", "clustered"])
def test_against_the_oracle(ctx, O, p, polydeg, n, kind):
    X = _nodes(kind, n + p)
    k = 2
    print(f"null-space solve p={p} deg={polydeg} n={n} {kind}", flush=True)
    st, _ = O.knn(X, X, n)
    col, vals, status = _weights(ctx, X, st, p, polydeg, OPS, k)
    assert not status.any()
    opl = [(O.OP_NAMES[o], k if o in ("Dxk", "Dyk") else 0) for o in OPS]
    Wq, _, _ = O.weights(X, X, st, None, p, polydeg, opl, quad=True)
    Wl, _, _ = O.weights(X, X, st, None, p, polydeg, opl, solve="lu")
    order = np.argsort(st, axis=1, kind="stable")
    assert np.array_equal(col, np.take_along_axis(st, order, 1))
    for o, name in enumerate(OPS):
        q = np.take_along_axis(Wq[:, o, :], order, 1)
        scale = np.abs(q).max(axis=1)
        e = np.abs(vals[o] - q).max(axis=1) / scale
        lu = np.abs(np.take_along_axis(Wl[:, o, :], order, 1) - q).max(axis=1) / scale
        print(f"  {name}: max {e.max():.2e} median {np.median(e):.2e} (LU {lu.max():.2e} {np.median(lu):.2e})",
              flush=True)
        assert e.max() <= max(1e-10, 4 * lu.max())
        assert np.median(e) <= max(1e-13, 2 * np.median(lu))


@pytest.mark.parametrize("p,polydeg,n", [(3, 3, 20), (7, 4, 31), (5, 5, 42), (9, 6, 57)])
@pytest.mark.parametrize("nops", [1, 2, 7])
def test_handed_back_rows(ctx, O, p, polydeg, n, nops, monkeypatch):
    """Rows whose stencil holds a duplicated or nearly duplicated node or a NaN
    get what the pivoting kernel alone gives them, bits and status; the other
    rows agree to rounding."""
    X = jittered_grid(24, 22, 0.25, seed=n)
    h = 1.0 / 23
    extra = X[[100, 260]].copy()                      # two exact duplicates
    near = X[[150, 400, 410]] + h * np.array([[1e-9, 0], [0, 1e-11], [3e-13, 1e-13]])
    X = np.concatenate([X, extra, near])
    st, _ = O.knn(X, X, n)
    Xn = X.copy()
    Xn[30, 1] = np.nan                                # after the search: its stencils carry a NaN
    ops = OPS[1:1 + nops] if nops < 7 else OPS
    print(f"handed-back rows p={p} n={n}, {nops} operators", flush=True)
    hit = np.isin(st, [100, 260, len(X) - 5, len(X) - 4]).sum(axis=1) > 0
    touched = np.isin(st, [30, 100, 260, 150, 400, 410] + list(range(len(X) - 5, len(X)))).any(axis=1)
    col, vals, status = _weights(ctx, Xn, st, p, polydeg, ops, 2)
    monkeypatch.setenv("RBFFD_NULLSPACE", "0")
    col0, vals0, status0 = _weights(ctx, Xn, st, p, polydeg, ops, 2)
    assert np.array_equal(col, col0)
    assert np.array_equal(status, status0)
    assert status[np.isin(st, [30]).any(axis=1)].all() and hit.any()
    for a, b in zip(vals, vals0):
        ok = ~touched
        d = np.abs(a[ok] - b[ok]).max(axis=1) / np.abs(b[ok]).max(axis=1)
        assert d.max() <= 1e-9
        bad = status0 != 0
        assert np.array_equal(a[bad], b[bad], equal_nan=True)


# sizes between the compiled ones: the edges of each kernel (11..22 nodes with 6
# monomials, 13..26 and 27..42 with 10, 18..31 and 32..47 with 15, 28..53 with 21)
BETWEEN = [(5, 2, 11), (5, 2, 22), (5, 3, 13), (5, 3, 26), (5, 3, 27), (7, 3, 42), (7, 4, 18), (7, 4, 30), (7, 4, 32),
           (9, 4, 47), (9, 5, 28), (9, 5, 53)]


@pytest.mark.parametrize("p,polydeg,n", BETWEEN)
@pytest.mark.parametrize("kind", ["grid", "clustered"])
def test_sizes_between_against_the_oracle(ctx, O, p, polydeg, n, kind):
    test_against_the_oracle(ctx, O, p, polydeg, n, kind)


# 48, 64 and 96 padded equations in the kernel that takes the rows handed back
@pytest.mark.parametrize("p,polydeg,n", [(5, 2, 17), (5, 3, 25), (5, 3, 38), (7, 4, 47), (9, 5, 53)])
@pytest.mark.parametrize("nops", [1, 2, 7])
def test_sizes_between_handed_back_rows(ctx, O, p, polydeg, n, nops, monkeypatch):
    test_handed_back_rows(ctx, O, p, polydeg, n, nops, monkeypatch)


@pytest.mark.parametrize("p,polydeg,n", [(5, 2, 17), (5, 3, 25), (5, 3, 35), (9, 5, 31)])
def test_sizes_between_grouped_rows(ctx, O, p, polydeg, n, monkeypatch):
    """Output rows that share stencils, up to 40 to one (more than a task
    holds), against the pivoting kernels; one call of single rows gives the bits
    of the grouped ones."""
    import rbffd_amd

    X = jittered_grid(17, 15, 0.25, seed=n)
    rng = np.random.default_rng(n)
    y2x = np.concatenate([np.full(40, 7), rng.integers(0, len(X), 500)]).astype(np.int32)
    Y = X[y2x] + rng.uniform(-0.02, 0.02, (len(y2x), 2))
    st, _ = O.knn(X, X, n)
    print(f"grouped rows p={p} deg={polydeg} n={n}", flush=True)
    eng = rbffd_amd.Engine(ctx)
    Xd, Yd, std = (ctx.to_device(a) for a in (X, Y, st.astype(np.int32)))

    def run():
        col, vals, status = eng.weights(Xd, Yd, std, ctx.to_device(y2x), p, polydeg, ["Dx", "Lap"], k=0)
        return col.get(), [v.get() for v in vals], status.get()

    col, vals, status = run()
    sd, Y1 = ctx.to_device(st[y2x].astype(np.int32)), Yd
    _, single, _ = eng.weights(Xd, Y1, sd, None, p, polydeg, ["Dx", "Lap"], k=0)
    single = [v.get() for v in single]
    monkeypatch.setenv("RBFFD_NULLSPACE", "0")
    col0, vals0, status0 = run()
    assert np.array_equal(col, col0) and not status.any() and not status0.any()
    for a, b, c in zip(vals, vals0, single):
        assert (np.abs(a - b).max(axis=1) <= 1e-9 * np.abs(b).max(axis=1)).all()
        assert np.array_equal(a, c)


# outside of it: fewer nodes or more than a kernel takes, a degree further above (m - 1) / 2, m = 3, even m
@pytest.mark.parametrize("p,polydeg,n", [(5, 2, 10), (5, 3, 43), (3, 2, 18), (3, 3, 25), (5, 4, 25), (6, 3, 25), (9, 5, 27), (3, 1, 10)])
def test_sizes_that_stay(ctx, O, p, polydeg, n, monkeypatch):
    X = jittered_grid(16, 15, 0.25, seed=n)
    st, _ = O.knn(X, X, n)
    print(f"sizes that stay p={p} deg={polydeg} n={n}", flush=True)
    col, vals, status = _weights(ctx, X, st, p, polydeg, ["Dx", "Lap"], 0)
    monkeypatch.setenv("RBFFD_NULLSPACE", "0")
    col0, vals0, status0 = _weights(ctx, X, st, p, polydeg, ["Dx", "Lap"], 0)
    assert np.array_equal(col, col0) and np.array_equal(status, status0)
    for a, b in zip(vals, vals0):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("p,polydeg,n,lines", [(3, 3, 20, 3), (5, 3, 21, 3), (5, 3, 25, 3), (7, 4, 31, 4), (7, 4, 39, 4),
                                               (7, 5, 43, 5), (9, 6, 57, 6), (9, 6, 57, 5)])
@pytest.mark.parametrize("method", [1, 3])
@pytest.mark.parametrize("diagonal", [False, True])
def test_dependent_monomials(O, p, polydeg, n, lines, method, diagonal, monkeypatch):
    """Nodes on at most as many straight lines as the degree (coordinates exact in
    binary): a polynomial of the basis vanishes on every stencil, so the monomial
    block is rank deficient up to rounding and each row is the pivoting kernel's,
    bit for bit.  Dx along the lines is determined all the same.  The eliminations
    of the sizes between keep it to 2e-11 in the median (the bar: 1e-9; a panel
    pivot of rounding left 1e-1 in the worst tenth of the rows); those of the
    compiled sizes, which take the monomials first, do not."""
    import rbffd_amd

    rng = np.random.default_rng(n + lines)
    nx = 2 * n
    x = np.round((np.arange(nx) + rng.uniform(-0.25, 0.25, (lines, nx))) * 2.0**14) / 2.0**20
    X = np.stack([x, np.broadcast_to(np.arange(lines)[:, None] / 64.0, x.shape)], -1).reshape(-1, 2)
    if diagonal:
        X = np.stack([X[:, 0] + X[:, 1], X[:, 1] - X[:, 0]], -1)
    st, _ = O.knn(X, X, n)
    ops = ["Dx", "Dxx", "Lap"]
    print(f"dependent monomials p={p} deg={polydeg} n={n} method={method} diagonal={diagonal}", flush=True)
    c = rbffd_amd.Context(0)  # no layout chosen by earlier, larger calls
    col, vals, status = _weights(c, X, st, p, polydeg, ops, 0, method=method)
    monkeypatch.setenv("RBFFD_NULLSPACE", "0")
    col0, vals0, status0 = _weights(c, X, st, p, polydeg, ops, 0, method=method)
    c.close()
    assert np.array_equal(col, col0) and np.array_equal(status, status0)
    for a, b in zip(vals, vals0):
        assert np.array_equal(a, b, equal_nan=True)
    if method == 1 and not diagonal and n in (25, 39):
        W, _, _ = O.weights(X, X, st, None, p, polydeg, [(O.OP_NAMES["Dx"], 0)], quad=True)
        q = np.take_along_axis(W[:, 0], np.argsort(st, axis=1, kind="stable"), 1)
        ok = (status == 0) & np.isfinite(q).all(axis=1)
        e = np.abs(vals[0] - q)[ok].max(axis=1) / np.abs(q)[ok].max(axis=1)
        assert np.quantile(e, 0.9) <= 1e-9


@pytest.mark.parametrize("p,polydeg,n", [(1, 3, 20), (3, 3, 20), (3, 4, 31), (3, 5, 42), (5, 5, 42), (5, 2, 18), (5, 3, 25),
                                         (5, 3, 35), (5, 3, 40), (7, 4, 37), (9, 5, 47), (1, 4, 31), (3, 6, 57)])
def test_rounding_against_the_elimination(ctx, O, p, polydeg, n, monkeypatch):
    """The weights' errors against 113 bits are no larger than the elimination's:
    the geometric mean over a jittered grid's rows and five operators.  The two
    differ per row by a factor whose logarithm has a deviation of about 0.5, so
    the mean over 1,225 rows (operators correlated) is known to 1.5%: the bar is
    1.015.  The last two shapes go to the elimination and give its bits."""
    X = jittered_grid(35, 35, 0.25, seed=n + p)
    ops = ["Dx", "Dy", "Dxx", "Dxy", "Lap"]
    st, _ = O.knn(X, X, n)
    W, _, _ = O.weights(X, X, st, None, p, polydeg, [(O.OP_NAMES[o], 0) for o in ops], quad=True)
    order = np.argsort(st, axis=1, kind="stable")
    col, vals, status = _weights(ctx, X, st, p, polydeg, ops, 0)
    monkeypatch.setenv("RBFFD_NULLSPACE", "0")
    col0, vals0, status0 = _weights(ctx, X, st, p, polydeg, ops, 0)
    assert np.array_equal(col, col0) and not status.any() and not status0.any()
    if polydeg > p + 2:
        assert all(np.array_equal(a, b) for a, b in zip(vals, vals0))
        return

    def err(v):
        e = []
        for o in range(len(ops)):
            q = np.take_along_axis(W[:, o], order, 1)
            e.append(np.abs(v[o] - q).max(axis=1) / np.abs(q).max(axis=1))
        return np.exp(np.log(np.maximum(e, 1e-18)).mean())

    print(f"p={p} deg={polydeg} n={n}: {err(vals):.2e}, elimination {err(vals0):.2e}", flush=True)
    assert err(vals) <= 1.015 * err(vals0)


@pytest.mark.parametrize("p,polydeg,n", [(3, 3, 20), (7, 4, 31), (3, 5, 42), (9, 6, 57), (5, 3, 25), (5, 3, 35), (9, 5, 47)])
@pytest.mark.parametrize("gap", [1e-9, 1e-11, 3e-13])
def test_near_duplicates_are_handed_back(O, p, polydeg, n, gap, monkeypatch):
    """Two nodes a small part of the spacing apart leave a pivot of S of about
    gap^m of the largest, far below the threshold: every row whose stencil holds
    both gets the pivoting kernel's bits.  Elsewhere the null-space solve ran: its
    rounding differs from that kernel's in nearly every row."""
    import rbffd_amd

    X = jittered_grid(24, 22, 0.25, seed=n)
    at = [150, 300, 410]
    X = np.concatenate([X, X[at] + gap / 23 * np.array([[1, 0], [0, 1], [0.6, -0.8]])])
    st, _ = O.knn(X, X, n)
    near = np.zeros(len(X), bool)
    for i, k in enumerate(at):
        near |= (st == k).any(axis=1) & (st == len(X) - 3 + i).any(axis=1)
    print(f"near duplicates p={p} deg={polydeg} n={n} gap={gap}: {near.sum()} rows", flush=True)
    c = rbffd_amd.Context(0)  # no layout chosen by earlier, larger calls
    ops = ["Dx", "Dyy", "Lap"]
    col, vals, status = _weights(c, X, st, p, polydeg, ops, 0)
    monkeypatch.setenv("RBFFD_NULLSPACE", "0")
    col0, vals0, status0 = _weights(c, X, st, p, polydeg, ops, 0)
    c.close()
    assert np.array_equal(col, col0) and np.array_equal(status, status0)
    assert near.sum() >= n
    for a, b in zip(vals, vals0):
        assert np.array_equal(a[near], b[near], equal_nan=True)
        assert (a != b).any(axis=1)[~near].mean() > 0.9


# low powers with high degrees: the split residual
@pytest.mark.parametrize("p,polydeg,n", [(1, 3, 20), (3, 4, 31), (5, 4, 31), (3, 5, 42), (3, 5, 43), (5, 6, 57)])
@pytest.mark.parametrize("kind", ["grid", "uniform", "clustered"])
def test_high_degrees_against_the_oracle(ctx, O, p, polydeg, n, kind):
    test_against_the_oracle(ctx, O, p, polydeg, n, kind)


@pytest.mark.parametrize("p,polydeg,n", [(3, 3, 20), (7, 4, 31), (3, 5, 42), (7, 5, 43), (9, 6, 57)])
def test_compiled_sizes_grouped_rows(ctx, O, p, polydeg, n, monkeypatch):
    test_sizes_between_grouped_rows(ctx, O, p, polydeg, n, monkeypatch)


@pytest.mark.parametrize("p,polydeg,n", [(3, 3, 20), (7, 4, 31), (7, 5, 43), (9, 6, 57), (5, 3, 25), (5, 3, 35)])
@pytest.mark.parametrize("unit", [2.0**-8, 1.0, 2.0**11])
def test_unscaled_frames(O, p, polydeg, n, unit, monkeypatch):
    """Method 3 solves in the nodes' own unit: the null-space solve runs whatever
    that is (its bits are not the pivoting kernel's in nearly every row), and the
    two agree to a few times the rounding of an FP64 solve at this conditioning
    (9e-9 at n = 57)."""
    import rbffd_amd

    X = unit * jittered_grid(23, 21, 0.25, seed=n)
    st, _ = O.knn(X, X, n)
    print(f"unscaled frames p={p} deg={polydeg} n={n} unit={unit}", flush=True)
    c = rbffd_amd.Context(0)  # no layout chosen by earlier, larger calls
    col, vals, status = _weights(c, X, st, p, polydeg, ["Dx", "Lap"], 0, method=3)
    monkeypatch.setenv("RBFFD_NULLSPACE", "0")
    col0, vals0, status0 = _weights(c, X, st, p, polydeg, ["Dx", "Lap"], 0, method=3)
    c.close()
    assert np.array_equal(col, col0) and not status.any() and not status0.any()
    for a, b in zip(vals, vals0):
        assert (a != b).any(axis=1).mean() > 0.9
        assert (np.abs(a - b).max(axis=1) <= (2e-8 if n == 57 else 1e-9) * np.abs(b).max(axis=1)).all()
