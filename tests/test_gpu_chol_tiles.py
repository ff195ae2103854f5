"""Cholesky for 64 < n <= 512: orders at the edges of the 32-column blocks, the
16-row tiles and the four kernels' ranges, padded leading dimensions with NaN,
both triangles, and factorizations that stop at the first, a middle and the last
column of a block.  The factor is the oracle's bits (the same fused
multiply-adds in the same order): the tolerance is zero."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("n", [65, 95, 97, 128, 129, 160, 191, 193, 256, 257, 481, 511, 512])
def test_potrf_tiles(queue, oracle, n, uplo):
    import magma_amd as ma
    rng = np.random.default_rng(n)
    count, ld = 6, n + n % 3
    F = rng.standard_normal((count, n, n))
    A = F @ F.transpose(0, 2, 1) + n * np.eye(n)
    fails = [0, 0, 0, 1, 32 + n % 31, n]            # info wanted; 0: none
    for s, f in enumerate(fails):
        if f:
            A[s, f - 1, f - 1] = -1.0 if s % 2 else np.nan
    keep = np.tril(np.ones((n, n), bool)) if uplo == "L" else np.triu(np.ones((n, n), bool))
    Ain = np.where(keep.T, A, np.nan)               # storage (column, row)
    print(f"potrf tiles n={n} uplo={uplo}", flush=True)
    dA = ma.DeviceBatch(Ain, ld=ld)
    if ld > n:
        dA.t[:, :, n:] = np.nan
    ret, info = ma.dpotrf_batched(dA, queue, uplo=ma.MagmaLower if uplo == "L" else ma.MagmaUpper)
    assert ret == 0
    assert list(info.cpu().numpy()) == fails
    got = dA.numpy()
    for s, f in enumerate(fails):
        k = f - 1 if f else n
        Lo, info_o = oracle.dpotrf(A[s], uplo=uplo.encode())
        assert info_o == f
        assert np.array_equal(got[s][:k, :k][keep.T[:k, :k]], Lo[:k, :k][keep.T[:k, :k]]), s
        assert np.isnan(got[s][~keep.T]).all(), s   # the other triangle is not written
