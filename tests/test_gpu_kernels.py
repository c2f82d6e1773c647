"""Single kernels of the library at the sizes where their tilings and splits can
go wrong, against LAPACK (scipy / the oracle) or plain numpy."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [64, 128, 192, 448, 8256])
def test_panel_pivot_choice(wm, ctx, oracle, prec, n):
    """The pivot is the lowest row among those of largest |re| + |im|, also when the
    candidates differ in their last bits only (equal high words) or are equal, in
    clusters of one workgroup, of several, and of more than 128 row blocks."""
    rng = np.random.RandomState(n)
    A = np.empty((1, n, n), np.complex128 if prec == "f64" else np.complex64)
    A[0] = rng.randn(n, n) + 1j * rng.randn(n, n)
    bits = rng.randint(0, 1000, n)
    top = np.sort(rng.choice(n, 3, replace=False))
    bits[top] = 1000  # three equal largest entries
    A[0, :, 0] = 4.0 + bits * (2.0 ** -50 if prec == "f64" else 2.0 ** -21)
    dev, piv, info = wm.getrf_batched(ctx, A, prec)
    P = piv.download()[0]
    assert info[0] == 0
    assert P[0] == top[0] + 1
    if n <= 448 and prec == "f64":
        assert np.array_equal(P, oracle.zgetrf(A[0])[1])
    B = rng.randn(n, 2) + 1j * rng.randn(n, 2)
    X = wm.getrs_batched(ctx, dev, piv, B, prec)[0]
    r = np.abs(A[0].astype(np.complex128) @ X - B).max() / (np.abs(A[0]).sum(axis=1).max() * np.abs(X).max())
    # partial pivoting on random entries: far below n^(2/3) growth times the unit roundoff
    assert r <= n ** (2 / 3) * (2.0 ** -53 if prec == "f64" else 2.0 ** -24), r


@pytest.mark.parametrize("n", [64, 256])
def test_panel_non_finite_entries(wm, ctx, n):
    """A NaN row is never a pivot candidate: the factorization ends and reports a zero
    pivot in the last column, where only that row is left; an all-NaN matrix reports the first."""
    rng = np.random.RandomState(n)
    A = rng.randn(2, n, n) + 1j * rng.randn(2, n, n)
    A[0, n // 3, 0] = np.nan
    A[1] = np.nan
    _, piv, info = wm.getrf_batched(ctx, A, "f64")
    assert list(info) == [n, 1]
    P = piv.download()
    assert np.all(P >= np.arange(1, n + 1)) and np.all(P <= n)


@pytest.mark.parametrize("ienv", [1, 2])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 128, 129, 700])
def test_fill_row_runs(wm, geometries, oracle, ctx, geo_dir, n, ienv):
    """Fills whose rows end inside, at and just beyond a run of 64 observation points and
    the padded size, for chains of segments (a dipole or monopole) and, at 700, a mesh
    with junctions: every entry against the oracle, the padding the identity."""
    import os
    p = os.path.join(geo_dir, f"runs_{n}_{ienv}.geo")
    if n >= 700:
        # with the ground each of the four rods gains a basis at its foot
        geometries.lightning(p, n - 4 if ienv == 2 else n, depth=0.0 if ienv == 2 else 0.5, ring=ienv == 1)
    elif ienv == 2:
        geometries.monopole(p, n)
    else:
        geometries.dipole(p, n + 1, 1.0, 0.2 / (n + 1))
    g = wm.Geometry.load(ctx, p, ienv=ienv)
    assert g.npls == n
    f = [5.0, 150.0]
    Z = g.fill(f)
    t = oracle.load(p, ienv=ienv)
    for i in range(2):
        ref = oracle.zmatrix(t, wm.wavenumber(f[i]), ienv=ienv)
        assert np.abs(Z[i] - ref).max() <= 1e-12 * np.abs(ref).max()
    import ctypes as C
    ka = np.array([wm.wavenumber(x) for x in f])
    D = wm.DeviceArray(ctx, np.full((2, g.ld, g.ld), np.nan, np.complex128))
    assert wm.lib().wm_zfill(ctx.h, g.h, 2, ka.ctypes.data_as(C.POINTER(C.c_double)), D.ptr, g.ld ** 2, None, 0) == 0
    full = D.download().transpose(0, 2, 1)
    assert np.array_equal(full[:, :n, :n], Z)
    eye = np.eye(g.ld)
    assert np.array_equal(full[:, n:], np.stack([eye[n:]] * 2)) and np.array_equal(full[:, :, n:], np.stack([eye[:, n:]] * 2))


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,batch", [(320, 70), (64, 5)])
def test_wide_batch_equals_single(wm, ctx, prec, n, batch):
    """A batch wide enough for the launches' larger tiles gives each member's factors and
    pivots bit for bit as factored alone (smaller tiles)."""
    rng = np.random.RandomState(n + batch)
    A = rng.randn(batch, n, n) + 1j * rng.randn(batch, n, n)
    dev, piv, info = wm.getrf_batched(ctx, A, prec)
    LU, P = dev.download(), piv.download()
    assert not info.any()
    for b in (0, batch // 2, batch - 1):
        d1, p1, _ = wm.getrf_batched(ctx, A[b], prec)
        assert np.array_equal(p1.download()[0], P[b])
        assert np.array_equal(d1.download()[0], LU[b])


@pytest.mark.parametrize("prec", ["f64", "f32", "bf16x3"])
@pytest.mark.parametrize("n,batch", [(8192, 1), (4160, 4)])
def test_lookahead_matches_one_stream(wm, ctx, prec, n, batch):
    """Factorizations large enough for the look-ahead stream, captured and launched directly,
    give the factors and pivots of the one-stream order (which the profiler keeps) bit for bit;
    captures are replayed with other work and synchronizations in between."""
    rng = np.random.RandomState(n)
    A = np.empty((batch, n, n), np.complex64 if prec != "f64" else np.complex128)
    for b in range(batch):
        A[b].real = rng.standard_normal((n, n))
        A[b].imag = rng.standard_normal((n, n))
    host = np.ascontiguousarray(A.transpose(0, 2, 1))
    dev, piv, _ = wm.getrf_batched(ctx, A, prec)

    def factor():
        import ctypes as C
        dev.upload(host)
        info = np.zeros(batch, np.int32)
        rc = wm.lib().wm_getrf_batched(ctx.h, wm.PREC_NAMES[prec], n, dev.ptr, n, n * n, piv.ptr, n, batch,
                                       info.ctypes.data_as(C.POINTER(C.c_int)))
        assert rc == 0
        return dev.download(), piv.download()

    ctx.prof_enable(True)
    ref = factor()
    ctx.prof_enable(False)
    for _ in range(2):  # replays
        got = factor()
        assert np.array_equal(got[1], ref[1]) and np.array_equal(got[0], ref[0])
    ctx.set_graphs(False)
    try:
        got = factor()
    finally:
        ctx.set_graphs(True)
    assert np.array_equal(got[1], ref[1]) and np.array_equal(got[0], ref[0])


@pytest.mark.parametrize("n", [64, 128, 192, 1024])
def test_preconditioner_solve_widths(wm, ctx, n):
    """The preconditioner's solves at every way their products are formed (up to
    4, up to 8 and up to 16 columns, then a second member), from one row block
    up.  Diagonally dominant matrices: 1e-12 of numpy's solution; a column has
    the same bits in every width; a column of NaN and one of infinities leave
    their neighbours alone."""
    L = wm.lib()
    L.wmx_getrs_grouped.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_void_p, C.c_int, C.c_void_p,
                                    C.c_void_p, C.c_int64, C.c_int, C.c_void_p, C.c_void_p, C.c_int, C.c_int]
    rng = np.random.RandomState(n)
    A = rng.randn(1, n, n) + 1j * rng.randn(1, n, n) + 4 * n ** 0.5 * np.eye(n)
    V = rng.randn(17, n) + 1j * rng.randn(17, n)
    dev, piv, info = wm.getrf_batched(ctx, A, "f64")
    assert not info.any()

    def solve(V, cols):
        Vd = wm.DeviceArray(ctx, np.ascontiguousarray(V))
        it, fac = np.array(cols, np.int32), np.zeros(len(cols), np.int32)
        assert L.wmx_getrs_grouped(ctx.h, wm.PREC_F64, n, 1, dev.ptr, 1, piv.ptr, Vd.ptr, n, len(it),
                                   it.ctypes.data, fac.ctypes.data, 1, 0) == 0
        out = Vd.download()
        Vd.free()
        return out

    ref = solve(V, range(17))
    x = np.linalg.solve(A[0], V.T).T
    assert np.abs(ref - x).max() <= 1e-12 * np.abs(x).max()
    for w in (1, 3, 4, 5, 8, 9, 16):
        got = solve(V, range(w))
        assert np.array_equal(got[:w].view(np.uint64), ref[:w].view(np.uint64)), w
        assert np.array_equal(got[w:].view(np.uint64), V[w:].view(np.uint64)), w
    for w in (4, 8, 16):
        bad = V.copy()
        bad[0, n // 2] = np.nan
        bad[w - 1, 0] = np.inf
        got = solve(bad, range(w))
        assert np.array_equal(got[1:w - 1].view(np.uint64), ref[1:w - 1].view(np.uint64)), w
        assert not np.isfinite(got[0]).all() and not np.isfinite(got[w - 1]).all()
    dev.free()
    piv.free()


@pytest.mark.parametrize("n", [64, 448, 512, 576, 640, 1088, 8192])
@pytest.mark.parametrize("noalloc", [False, True])
def test_row_permutation(wm, ctx, n, noalloc):
    """The interchanges of a pivot sequence applied to a right-hand side (factors:
    the identity, so the solution is the permuted vector, exactly): sequences of
    a factorization (row i meets a row at or below it) and any others, at sizes
    of one part, of parts that are empty, ragged or whole."""
    rng = np.random.RandomState(n)
    A = wm.DeviceArray(ctx, np.ascontiguousarray(np.broadcast_to(np.eye(n, dtype=np.complex128), (2, n, n))))
    piv = np.empty((2, n), np.int32)
    piv[0] = [rng.randint(i, n) + 1 for i in range(n)]
    piv[1] = rng.randint(0, n, n) + 1
    P = wm.DeviceArray(ctx, piv)
    b = np.arange(2 * n, dtype=np.complex128).reshape(2, 1, n)
    B = wm.DeviceArray(ctx, b)
    f = wm.lib().wm_getrs_batched_noalloc if noalloc else wm.lib().wm_getrs_batched
    assert f(ctx.h, wm.PREC_F64, n, 1, A.ptr, n, C.c_int64(n * n), P.ptr, C.c_int64(n),
             B.ptr, n, C.c_int64(n), 2) == 0
    ref = b.copy()
    for m in range(2):
        for i in range(n):
            p = piv[m, i] - 1
            ref[m, 0, [i, p]] = ref[m, 0, [p, i]]
    assert np.array_equal(B.download(), ref)
    for d in (A, P, B):
        d.free()


@pytest.mark.parametrize("n", [2, 127, 128, 2100])
def test_host_matrices(wm, geometries, ctx, geo_dir, n):
    """Matrices to and from the host where the device pads them: a few rows, no padding
    (128), and 2100 rows (two chunks).  zmatrix equals the batched fill's values
    bit for bit, and LU_cuBLAS solves with the matrix it is given (residual within
    n eps of |A| |x|, as partial pivoting gives on random matrices)."""
    import os
    p = os.path.join(geo_dir, f"host_{n}.geo")
    geometries.dipole(p, n + 1, 1.0, 0.2 / (n + 1))
    Z = wm.zmatrix(wm.configwire(p), wm.wavenumber(150.0))
    assert Z.shape == (n, n)
    assert np.array_equal(Z, wm.Geometry.load(ctx, p).fill([150.0])[0])
    rng = np.random.RandomState(n)
    A = rng.randn(n, n) + 1j * rng.randn(n, n)
    b = rng.randn(n, 3) + 1j * rng.randn(n, 3)
    x = wm.LU_cuBLAS(A, b)
    r = np.abs(A @ x - b).max() / (np.abs(A).sum(axis=1).max() * np.abs(x).max())
    assert r <= n * 2.0 ** -52


@pytest.mark.parametrize("prec,rows", [("f64", 128), ("f32", 256)])
@pytest.mark.parametrize("n", [256, 1024, 1088])
def test_panel_fewer_parts(wm, ctx, prec, rows, n):
    """A matrix whose clusters do not fit at the usual rows per workgroup is factored
    with half the parts per row and twice the rows: the same factors and pivots,
    bit for bit; one workgroup less, and it is refused."""
    L = wm.lib()
    L.wmx_set_panel_resident.argtypes = [C.c_void_p, C.c_int]
    rng = np.random.RandomState(n)
    A = rng.randn(2, n, n) + 1j * rng.randn(2, n, n)
    dev, piv, info = wm.getrf_batched(ctx, A, prec)
    ref, P = dev.download(), piv.download()
    assert not info.any()
    cap = -(-n // rows)
    assert L.wmx_set_panel_resident(ctx.h, cap) == 0
    try:
        dev, piv, info = wm.getrf_batched(ctx, A, prec)
        assert not info.any()
        assert np.array_equal(piv.download(), P)
        assert np.array_equal(dev.download(), ref)
        if cap > 1:
            assert L.wmx_set_panel_resident(ctx.h, cap - 1) == 0
            with pytest.raises(wm.WireMoMError):
                wm.getrf_batched(ctx, A, prec)
    finally:
        assert L.wmx_set_panel_resident(ctx.h, 0) == 0


def test_mixed_sweep_routes_by_model(wm, geometries, ctx, geo_dir):
    """A wide split-BF16x3 sweep of a size where the cost model takes FP64 factors gets them
    for every frequency, with the FP64 sweep's bits (the model by itself: the host tests)."""
    import os
    p = os.path.join(geo_dir, "route_2048.geo")
    geometries.planar_grid(p, 2048, seed=3, size=5.0)
    g = wm.Geometry.load(ctx, p)
    f = np.linspace(20.0, 60.0, 63)
    zin, cur, st = wm.solve_sweep(g, f, [7], "bf16x3")
    assert [s["prec"] for s in st] == [wm.PREC_F64] * len(f)
    z64, c64, _ = wm.solve_sweep(g, f, [7], "f64")
    assert np.array_equal(zin, z64) and np.array_equal(cur, c64)


@pytest.mark.parametrize("prec,rows", [("f64", 128), ("f32", 256)])
@pytest.mark.parametrize("n", [192, 576, 8320])
def test_panel_tall(wm, ctx, prec, rows, n):
    """The panel of matrices too tall for the usual clusters, at partly filled workgroups and
    at more workgroups than a wave has lanes: factors, pivots and zero-pivot reports of the
    usual panel, bit for bit, on random entries, with a zero column and with a NaN row, for
    every member and through an index table, launched directly and replayed."""
    L = wm.lib()
    L.wmx_set_panel_resident.argtypes = [C.c_void_p, C.c_int]
    L.wmx_getrf_batched_idx.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_void_p, C.c_int, C.c_int64, C.c_void_p,
                                        C.c_int64, C.c_int, C.c_void_p, C.c_void_p]
    rng = np.random.RandomState(n)
    b, p = 3 if n < 4096 else 1, wm.PREC_NAMES[prec]
    A = np.empty((b, n, n), np.complex128 if prec == "f64" else np.complex64)
    A.real = rng.standard_normal((b, n, n))
    A.imag = rng.standard_normal((b, n, n))
    if b > 1:
        A[1, n // 2] = 0.0  # members are stored column by column: a zero column
        A[2, :, n // 3] = np.nan
    dev = wm.DeviceArray(ctx, A)
    piv = wm.DeviceArray(ctx, np.zeros((b, n), np.int32))
    idx = np.arange(b, dtype=np.int32)[::-1].copy()

    def factor(indexed):
        dev.upload(A)
        piv.upload(np.zeros((b, n), np.int32))
        info = np.zeros(b, np.int32)
        if indexed:
            assert L.wmx_getrf_batched_idx(ctx.h, p, n, dev.ptr, n, n * n, piv.ptr, n, b, info.ctypes.data,
                                           idx.ctypes.data) == 0
            info = info[idx]
        else:
            assert L.wm_getrf_batched(ctx.h, p, n, dev.ptr, n, n * n, piv.ptr, n, b,
                                      info.ctypes.data_as(C.POINTER(C.c_int))) >= 0  # > 0: a zero pivot
        ctx.sync()
        return dev.download(), piv.download(), info

    ref = factor(False)
    if b > 1:
        assert ref[2][0] == 0 and ref[2][1] == n // 2 + 1 and ref[2][2] == n
    try:
        assert L.wmx_set_panel_resident(ctx.h, -(-n // rows)) == 0
        for graphs, indexed in ((True, False), (True, False), (False, True)):
            ctx.set_graphs(graphs)
            got = factor(indexed)
            assert np.array_equal(got[2], ref[2])
            assert np.array_equal(got[1], ref[1])
            assert np.array_equal(got[0], ref[0], equal_nan=True)
    finally:
        ctx.set_graphs(True)
        assert L.wmx_set_panel_resident(ctx.h, 0) == 0
    dev.free()
    piv.free()


@pytest.mark.parametrize("form", ["f64", "f32", "f64 noalloc", "f32 noalloc", "f64 transposed"])
@pytest.mark.parametrize("n", [64, 128, 192, 576])
def test_solve_widths(wm, ctx, n, form):
    """Triangular solves at every way their right-hand sides are divided: one launch member
    of up to 16 columns (both forms of the products, one or two columns per wave), two
    members of even and of uneven widths, and a second pass beyond 32.  Two matrices, a
    leading dimension above n.  The residual is a backward-stable solve's (n unit roundoffs
    of the factors' precision), each column has the bits of the same column solved by itself,
    and the rows between columns keep what they held."""
    prec, kind = form.split()[0], form.split()[-1]
    rng = np.random.RandomState(n)
    A = rng.randn(2, n, n) + 1j * rng.randn(2, n, n)
    dev, piv, info = wm.getrf_batched(ctx, A, prec)
    assert not info.any()
    A = A.astype(np.complex64 if prec == "f32" else np.complex128).astype(np.complex128)
    op = A.conj().transpose(0, 2, 1) if kind == "transposed" else A
    L, ld = wm.lib(), n + 5
    f = {"noalloc": L.wm_getrs_batched_noalloc, "transposed": L.wmx_getrs_trans}.get(kind, L.wm_getrs_batched)

    def solve(B):
        k = B.shape[1]
        pad = np.full((2, k, ld), 7.0 - 3.0j)
        pad[:, :, :n] = B
        D = wm.DeviceArray(ctx, pad)
        assert f(ctx.h, wm.PREC_NAMES[prec], n, k, dev.ptr, n, C.c_int64(n * n), piv.ptr,
                 C.c_int64(n), D.ptr, ld, C.c_int64(k * ld), 2) == 0
        ctx.sync()
        X = D.download()
        D.free()
        assert np.all(X[:, :, n:] == 7.0 - 3.0j)
        return X[:, :, :n]

    widths = {"transposed": (1, 9, 17)}.get(kind, (1, 4, 5, 8, 9, 15, 16, 17, 18, 31, 32, 33, 40))
    B = rng.randn(2, max(widths), n) + 1j * rng.randn(2, max(widths), n)
    alone = np.concatenate([solve(B[:, r:r + 1]) for r in range(max(widths))], axis=1)
    u = 2.0 ** (-24 if prec == "f32" else -53)
    R = np.matmul(alone, op.transpose(0, 2, 1)) - B
    assert np.abs(R).max() <= n * u * np.abs(op).sum(axis=2).max() * np.abs(alone).max()
    for k in widths:
        X = solve(B[:, :k])
        assert np.array_equal(X.view(np.uint64), alone[:, :k].copy().view(np.uint64)), k
    dev.free()
    piv.free()


def test_preconditioner_solve_grouping(wm, ctx):
    """The preconditioner's solves with several factors, items in another order than they are
    stored and members of 16, 4, 12 and 4 columns (20, 12 and 4 columns of three factors):
    1e-12 of numpy's solutions on diagonally dominant matrices, each item with the bits it
    has when solved by itself, and items outside the list untouched."""
    L = wm.lib()
    L.wmx_getrs_grouped.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_void_p, C.c_int, C.c_void_p,
                                    C.c_void_p, C.c_int64, C.c_int, C.c_void_p, C.c_void_p, C.c_int, C.c_int]
    rng = np.random.RandomState(11)
    n, nf, nr, nv = 192, 3, 4, 10
    A = rng.randn(nf, n, n) + 1j * rng.randn(nf, n, n) + 4 * n ** 0.5 * np.eye(n)
    V = rng.randn(nv, nr, n) + 1j * rng.randn(nv, nr, n)
    items = [8, 1, 2, 3, 4, 5, 6, 7, 0]  # item 9 takes no part
    fac = [0, 0, 1, 2, 0, 1, 0, 1, 0]
    dev, piv, info = wm.getrf_batched(ctx, A, "f64")
    assert not info.any()

    def solve(items, fac):
        Vd = wm.DeviceArray(ctx, V)
        it, f = np.array(items, np.int32), np.array(fac, np.int32)
        assert L.wmx_getrs_grouped(ctx.h, wm.PREC_F64, n, nr, dev.ptr, nf, piv.ptr, Vd.ptr, n * nr, len(it),
                                   it.ctypes.data, f.ctypes.data, 1, 0) == 0
        out = Vd.download()
        Vd.free()
        return out

    got = solve(items, fac)
    assert np.array_equal(got[9], V[9])
    for q, f in zip(items, fac):
        x = np.linalg.solve(A[f], V[q].T).T
        assert np.abs(got[q] - x).max() <= 1e-12 * np.abs(x).max()
        assert np.array_equal(solve([q], [f])[q].view(np.uint64), got[q].view(np.uint64))
    dev.free()
    piv.free()


@pytest.mark.parametrize("prec,n,cap", [("f64", 512, 8), ("f64", 512, 20), ("f32", 640, 5)])
def test_contexts_factor_side_by_side(wm, ctx, prec, n, cap):
    """Contexts of four threads on one device that take its panel workgroups to be so few that
    no two clusters fit (cap 8 or 5), or only two (20): every factorization gives the
    bits it gives alone, while contexts come and go."""
    import threading
    L = wm.lib()
    L.wmx_set_panel_resident.argtypes = [C.c_void_p, C.c_int]
    rng = np.random.RandomState(n)
    A = [rng.randn(3, n, n) + 1j * rng.randn(3, n, n) for _ in range(4)]
    ref = []
    for a in A:
        dev, piv, info = wm.getrf_batched(ctx, a, prec)
        assert not info.any()
        ref.append((dev.download(), piv.download()))
    bad = []

    def work(k):
        try:
            c = wm.Context(0)
            c.set_graphs(False)  # other threads drive the device
            assert L.wmx_set_panel_resident(c.h, cap) == 0
            for _ in range(8):
                dev, piv, info = wm.getrf_batched(c, A[k], prec)
                if info.any() or not (np.array_equal(dev.download(), ref[k][0]) and
                                      np.array_equal(piv.download(), ref[k][1])):
                    bad.append(k)
                dev.free()
                piv.free()
            c.close()
        except Exception as e:  # reported by the main thread
            bad.append((k, repr(e)))

    t = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for x in t:
        x.start()
    for _ in range(3):
        wm.Context(0).close()
    for x in t:
        x.join()
    assert not bad


@pytest.mark.parametrize("ienv", [1, 2])
def test_fill_peaks_off_their_segments(wm, geometries, oracle, ctx, geo_dir, ienv):
    """Bases whose peak is not a node of their segments (arrays a caller may pass): halves of
    one segment then have several observation points, which the row tables keep apart, within
    a run of rows and from run to run.  Every entry against the oracle."""
    import os
    p = os.path.join(geo_dir, f"peaks_{ienv}.geo")
    (geometries.monopole if ienv == 2 else geometries.dipole)(p, *((300,) if ienv == 2 else (301, 1.0, 0.0005)))
    t, o = wm.configwire(p, ienv=ienv), oracle.load(p, ienv=ienv)
    n = t.npls
    rng = np.random.RandomState(5)
    for b in rng.choice(np.arange(5, n - 5), 40, replace=False):
        # four nodes further along the wire: no half of zero length
        t.ipc[b] = o.ipc[b] = abs(int(t.ipc[b])) + 4
    g = wm.Geometry.from_topology(ctx, t, ienv)
    assert g.npls == n
    Z = g.fill([90.0])[0]
    ref = oracle.zmatrix(o, wm.wavenumber(90.0), ienv=ienv)
    assert np.abs(Z - ref).max() <= 1e-12 * np.abs(ref).max()
