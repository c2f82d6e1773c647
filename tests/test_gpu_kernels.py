"""Single kernels of the library at the sizes where their tilings and splits can
go wrong, against LAPACK (scipy / the oracle) or plain numpy."""
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
