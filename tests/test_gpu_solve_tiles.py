"""Solves with 16 right-hand sides in registers (n <= 512): orders and
right-hand-side counts at the edges of the 16-row tiles and of the kernels'
order ranges, pivots at random, leading dimensions above n with NaN in the
padding, and NaN in the triangle that a routine does not read."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [(1, 1), (15, 17), (16, 16), (17, 3), (48, 33), (63, 2), (64, 16), (65, 15), (127, 5), (128, 32), (129, 1),
         (192, 17), (255, 2), (256, 16), (257, 3), (300, 31), (511, 1), (512, 17)]


def same(a, b):
    a = np.asarray(a); b = np.asarray(b)
    return a.shape == b.shape and bool(np.all((a == b) | (np.isnan(a) & np.isnan(b))))


def factor_batch(rng, count, n):
    """LU factors of well-conditioned matrices with arbitrary interchanges."""
    LU = rng.uniform(-1, 1, (count, n, n)) / max(1.0, n / 8.0)
    LU[:, np.arange(n), np.arange(n)] = rng.uniform(1, 2, (count, n)) * rng.choice([-1.0, 1.0], (count, n))
    ipiv = np.stack([[rng.integers(k, n) + 1 for k in range(n)] for _ in range(count)]).astype(np.int32)
    return LU, ipiv


def device(A, ld, fill=np.nan):
    import magma_amd as ma
    d = ma.DeviceBatch(A, ld=ld)
    if ld > A.shape[2]:
        d.t[:, :, A.shape[2]:] = fill
    return d


@pytest.mark.parametrize("n,nrhs", CASES)
@pytest.mark.parametrize("trans", ["N", "T"])
def test_getrs_tiles(queue, oracle, n, nrhs, trans):
    """No-transpose bitwise the oracle's dgetrs; transposed by its residual."""
    import magma_amd as ma
    rng = np.random.default_rng(n * 100 + nrhs)
    count = 3
    LU, ipiv = factor_batch(rng, count, n)
    B = rng.uniform(-1, 1, (count, nrhs, n))
    B[1][:, n // 2:] = 0.0                     # zeros among the solved rows
    dA, dB = device(LU, n + 3), device(B, n + 5)
    ip = ma.IntBatch(count, n)
    ip.t.copy_(__import__("torch").from_numpy(ipiv))
    t = ma.MagmaNoTrans if trans == "N" else ma.MagmaTrans
    print(f"getrs tiles n={n} nrhs={nrhs} trans={trans}", flush=True)
    assert ma.dgetrs_batched(dA, ip, dB, queue, trans=t) == 0
    X = dB.numpy()
    assert bool(dB.t[:, :, n:].isnan().all())
    for s in range(count):
        if trans == "N":
            assert same(X[s], oracle.dgetrs(LU[s], ipiv[s], B[s])), s
        else:
            L = np.tril(LU[s].T, -1) + np.eye(n)
            A = L @ np.triu(LU[s].T)           # rows in pivot order
            for k in reversed(range(n)):
                p = ipiv[s][k] - 1
                A[[k, p]] = A[[p, k]]
            assert oracle.solve_error(A, X[s], B[s]) < 30, s      # storage of A' is A's rows


@pytest.mark.parametrize("n,nrhs", CASES)
@pytest.mark.parametrize("uplo", ["L", "U"])
def test_potrs_tiles(queue, oracle, n, nrhs, uplo):
    import magma_amd as ma
    rng = np.random.default_rng(n * 100 + nrhs + 1)
    count = 2
    F, _ = factor_batch(rng, count, n)
    F[:, np.arange(n), np.arange(n)] = np.abs(F[:, np.arange(n), np.arange(n)])
    L = np.stack([np.tril(f.T) for f in F])
    S = np.stack([m.T if uplo == "L" else m for m in L])          # storage[j, i] = factor(i, j)
    other = np.triu(np.ones((n, n), bool), 1)                     # never read
    S = np.where(other.T if uplo == "L" else other, np.nan, S)
    B = rng.uniform(-1, 1, (count, nrhs, n))
    dA, dB = device(S, n + 2), device(B, n + 1)
    print(f"potrs tiles n={n} nrhs={nrhs} uplo={uplo}", flush=True)
    assert ma.dpotrs_batched(dA, dB, queue, uplo=ma.MagmaLower if uplo == "L" else ma.MagmaUpper) == 0
    X = dB.numpy()
    for s in range(count):
        A = L[s] @ L[s].T
        assert oracle.solve_error(A, X[s], B[s]) < 30, s


@pytest.mark.parametrize("n", [40, 100, 256, 400])
def test_nonfinite_factor_falls_back(queue, oracle, n):
    """A zero x_k under an Inf multiplier or over a zero pivot is skipped, as
    reference dtrsm does, and the matrices beside it are unaffected."""
    import magma_amd as ma
    import torch
    rng = np.random.default_rng(n)
    LU, ipiv = factor_batch(rng, 4, n)
    ipiv[:] = np.arange(1, n + 1)
    B = rng.uniform(-1, 1, (4, 3, n))
    B[:, :, 0] = 0.0
    LU[1][0, 5] = np.inf                       # L(5, 0), x_0 = 0
    LU[2][n - 1, n - 1] = 0.0                  # U(n-1, n-1), x_{n-1} = 0 in column 0
    B[2][0, :] = 0.0
    LU[3][n // 2, n - 1] = np.nan              # a multiplier that is used
    dA, dB = device(LU, n), device(B, n)
    ip = ma.IntBatch(4, n)
    ip.t.copy_(torch.from_numpy(ipiv))
    assert ma.dgetrs_batched(dA, ip, dB, queue) == 0
    X = dB.numpy()
    for s in range(4):
        assert same(X[s], oracle.dgetrs(LU[s], ipiv[s], B[s])), s
    assert np.all(np.isfinite(X[1])) and np.all(np.isfinite(X[2][0]))
