"""Batched QR in registers (m, n <= 128): the edges of its row and column
tiles, operands near the ends of the exponent range and non-finite ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53


def run(queue, A, ld):
    import magma_amd as ma
    import torch
    count, n, m = A.shape
    dA = ma.DeviceBatch(A, ld=ld)
    tau = ma.DeviceBatch(np.full((count, 1, min(m, n)), 9.0))
    info = torch.full((count,), -1, dtype=torch.int32, device="cuda")
    ret = ma.load().magma_dgeqrf_batched(m, n, dA.ptr, dA.ld, tau.ptr, info.data_ptr(), count, queue.handle)
    assert ret == 0
    assert np.all(info.cpu().numpy() == 0)
    return dA, dA.numpy(), tau.numpy()[:, 0, :]


SHAPES = [(1, 3), (3, 1), (15, 16), (16, 17), (17, 16), (32, 31), (33, 16), (33, 32), (64, 16), (64, 17), (65, 32),
          (16, 64), (63, 64), (65, 33), (127, 32), (32, 127), (128, 128), (127, 65), (129, 5), (5, 129)]


@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("scale", [1.0, 1e-220, 1e180])
def test_tile_edges(queue, oracle, m, n, scale):
    """The tester's two residuals, and R and tau those of the oracle's dgeqr2
    to rounding; matrix 1 has a zero column, matrix 2 a subdiagonal of zeros
    (tau = 0 throughout), and nothing outside the m x n blocks is written."""
    rng = np.random.default_rng(1000 * m + n)
    A = rng.uniform(-1, 1, (4, n, m)) * scale
    A[1][n // 2, :] = 0.0
    A[2] = np.tril(A[2]) if n == m else A[2]        # storage is transposed: an upper triangular matrix
    dA, F, T = run(queue, A, m + 3)
    assert bool((dA.t[:, :, m:] == 0).all())
    k = min(m, n)
    for s in range(4):
        e1, e2 = oracle.qr_errors(A[s] / scale, np.where(np.triu(np.ones((m, n))).T > 0, F[s] / scale, F[s]), T[s], m, n)
        assert e1 < 30 * EPS and e2 < 30 * EPS, (s, e1, e2)
        Fo, to = oracle.dgeqrf(A[s])
        top = np.abs(Fo).max()
        assert np.abs(np.triu(F[s].T[:k, :]) - np.triu(Fo.T[:k, :])).max() <= 1e-12 * top * max(m, n), s
        assert np.abs(T[s] - to).max() <= 1e-12 * max(m, n), s
    if m == n:
        assert np.all(T[2] == 0.0) and np.array_equal(F[2], A[2])


@pytest.mark.parametrize("m,n", [(16, 16), (64, 64), (100, 100)])
def test_nonfinite_stays_in_its_columns(queue, oracle, m, n):
    """An Inf in the last column reaches no other column, and a NaN below the
    first row makes that column's tau NaN as dgeqr2 does."""
    rng = np.random.default_rng(m)
    A = rng.uniform(-1, 1, (2, n, m))
    A[0][n - 1, m // 2] = np.inf
    A[1][0, m - 1] = np.nan
    _, F, T = run(queue, A, m)
    _, Fr, Tr = run(queue, np.where(np.isfinite(A), A, 0.5), m)
    assert np.array_equal(F[0][: n - 1], Fr[0][: n - 1]) and np.array_equal(T[0][: n - 1], Tr[0][: n - 1])
    assert np.isnan(oracle.dgeqrf(A[1])[1][0]) and np.isnan(T[1][0])


@pytest.mark.parametrize("m,n", [(2, 2), (40, 40), (65, 33), (100, 100), (128, 7), (129, 129), (300, 3)])
def test_a_lone_nan_reaches_tau(queue, oracle, m, n):
    """A NaN that is all a column has below its diagonal, in the first column
    (matrix 0) and in the last one that has a reflector (1): tau and R are NaN
    exactly where dgeqr2's are."""
    rng = np.random.default_rng(m + n)
    k = min(m - 1, n) - 1
    A = np.stack([np.triu(rng.uniform(1, 2, (m, n))).T] * 2)        # storage is transposed
    A[0][0, m - 1] = np.nan
    A[1][k, k + 1] = np.nan
    print(f"geqrf nan m={m} n={n}", flush=True)
    _, F, T = run(queue, A, m)
    for s, i in enumerate((0, k)):
        Fo, to = oracle.dgeqrf(A[s])
        assert np.isnan(to[i]) and np.array_equal(np.isnan(T[s]), np.isnan(to)), s
        top = np.triu(np.ones((m, n), bool)).T
        assert np.array_equal(np.isnan(F[s][top]), np.isnan(Fo[top])), s
