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


TRSM = [(s, u, t) for s in "LR" for u in "UL" for t in "NT"]


@pytest.mark.parametrize("side,uplo,trans", TRSM)
@pytest.mark.parametrize("order,nv", [(15, 1), (16, 17), (17, 16), (63, 33), (65, 2), (128, 15), (129, 18), (250, 40),
                                      (257, 16), (512, 3)])
def test_trsm_tiles(queue, oracle, side, uplo, trans, order, nv):
    """Bitwise the oracle's dtrsm at the edges of the tiles and of the kernels'
    order ranges, unit and non-unit, with NaN where A is not read; matrix 2 has
    an Inf multiplier, taken or skipped as the reference loops do."""
    import magma_amd as ma
    L = ma.load()
    rng = np.random.default_rng(order * 10 + nv)
    m, n = (order, nv) if side == "L" else (nv, order)
    for diag, alpha in (("N", 1.0), ("U", -0.5)):
        F, _ = factor_batch(rng, 3, order)
        keep = np.tril(np.ones((order, order), bool), 0 if diag == "N" else -1)
        A = np.where(keep if uplo == "U" else keep.T, F, np.nan)       # storage is transposed
        B = rng.uniform(-1, 1, (3, n, m))
        B[1][:, : m // 2] = 0.0
        B[2][: n // 2 + 1, :] = 0.0
        if order > 5:
            A[2][(5, 2) if uplo == "U" else (2, 5)] = np.inf
        dA, dB = device(A, order + 1), device(B, m + 2)
        print(f"trsm tiles {side}{uplo}{trans}{diag} order={order} nv={nv}", flush=True)
        L.magmablas_dtrsm_batched(ma.MagmaLeft if side == "L" else ma.MagmaRight,
                                  ma.MagmaUpper if uplo == "U" else ma.MagmaLower,
                                  ma.MagmaNoTrans if trans == "N" else ma.MagmaTrans,
                                  ma.MagmaNonUnit if diag == "N" else ma.MagmaUnit, m, n, alpha, dA.ptr, dA.ld,
                                  dB.ptr, dB.ld, 3, queue.handle)
        X = dB.numpy()
        assert bool(dB.t[:, :, m:].isnan().all())
        for s in range(3):
            want = oracle.dtrsm(side.encode(), uplo.encode(), trans.encode(), diag.encode(), m, n, alpha, A[s], B[s])
            assert same(X[s], want), (diag, s)


@pytest.mark.parametrize("n", [2, 15, 17, 48, 63, 65, 127, 129, 200, 257, 511])
def test_getri_tiles(queue, oracle, n):
    """Bitwise the oracle's dgetrs on the identity; matrix 1 is singular."""
    import magma_amd as ma
    import torch
    rng = np.random.default_rng(n)
    LU, ipiv = factor_batch(rng, 2, n)
    LU[1][n // 2, n // 2] = 0.0
    dA, dI = device(LU, n + 1), ma.DeviceBatch(np.full((2, n, n), 7.0), ld=n + 2)
    ip = ma.IntBatch(2, n)
    ip.t.copy_(torch.from_numpy(ipiv))
    info = torch.full((2,), -1, dtype=torch.int32, device="cuda")
    print(f"getri tiles n={n}", flush=True)
    assert ma.load().magma_dgetri_outofplace_batched(n, dA.ptr, dA.ld, ip.ptr, dI.ptr, dI.ld, info.data_ptr(), 2,
                                                     queue.handle) == 0
    for s in range(2):
        assert same(dI.numpy()[s], oracle.dgetrs(LU[s], ipiv[s], np.eye(n))), s
    assert info.cpu().tolist() == [0, n // 2 + 1]


@pytest.mark.parametrize("n", [17, 27, 64, 65, 129, 257, 491])
def test_unread_values_do_not_leave_the_sweeps(queue, n):
    """With NaN in the padding and in the triangle that is not read, the solves
    stay with the register sweeps.  Only those turn zeros of a zero right-hand
    side over a negative diagonal into -0 (back, after potrs's second sweep): the reference loops, which
    a result that is not finite goes back to, skip a zero and keep its sign."""
    import magma_amd as ma
    import torch
    rng = np.random.default_rng(n)
    F, _ = factor_batch(rng, 2, n)
    F[:, np.arange(n), np.arange(n)] = -np.abs(F[:, np.arange(n), np.arange(n)])
    low = np.where(np.tril(np.ones((n, n), bool)).T, F, np.nan)        # storage is transposed
    B = rng.uniform(-1, 1, (2, 5, n))
    B[:, 2] = 0.0
    L = ma.load()
    for ld in (n, n + 3):
        print(f"sweeps n={n} ld={ld}", flush=True)
        dA, dB = device(low, ld), device(B, n)
        L.magmablas_dtrsm_batched(ma.MagmaLeft, ma.MagmaLower, ma.MagmaNoTrans, ma.MagmaNonUnit, n, 5, 1.0, dA.ptr,
                                  dA.ld, dB.ptr, dB.ld, 2, queue.handle)
        X = dB.numpy()
        assert np.isfinite(X).all() and (X[:, 2] == 0).all() and np.signbit(X[:, 2]).any(axis=1).all()
        dB = device(B, n)
        assert ma.dpotrs_batched(dA, dB, queue, uplo=ma.MagmaLower) == 0
        X = dB.numpy()
        assert np.isfinite(X).all() and (X[:, 2] == 0).all() and not np.signbit(X[:, 2, n - 1]).any()
        dA, dB = device(F, ld), device(B, n)
        ip = ma.IntBatch(2, n)
        ip.t.copy_(torch.arange(1, n + 1, dtype=torch.int32).repeat(2, 1))
        assert ma.dgetrs_batched(dA, ip, dB, queue) == 0
        X = dB.numpy()
        assert np.isfinite(X).all() and (X[:, 2] == 0).all() and np.signbit(X[:, 2]).any(axis=1).all()


@pytest.mark.parametrize("side,uplo,trans", [c for c in TRSM if c not in (("L", "L", "T"), ("R", "L", "N"))])
@pytest.mark.parametrize("count,nv,orders", [(4, 5, (6, 7, 11, 12, 14, 15)), (4200, 13, (8, 9, 13, 14, 17, 18)),
                                             (4200, 7, (11, 12, 15, 16, 20, 21)), (8300, 2, (24, 25, 28, 29, 40, 41))])
def test_trsm_lane_and_sweep(queue, oracle, side, uplo, trans, count, nv, orders):
    """Either side of the lines between the lane per vector and the sweeps:
    bitwise the oracle's dtrsm."""
    import magma_amd as ma
    rng = np.random.default_rng(count + nv)
    for order in orders:
        m, n = (order, nv) if side == "L" else (nv, order)
        F, _ = factor_batch(rng, 4, order)
        B = rng.uniform(-1, 1, (4, n, m))
        reps = -(-count // 4)
        dA, dB = device(np.tile(F, (reps, 1, 1))[:count], order), device(np.tile(B, (reps, 1, 1))[:count], m)
        print(f"trsm lanes/sweep {side}{uplo}{trans} order={order} nv={nv} count={count}", flush=True)
        ma.load().magmablas_dtrsm_batched(ma.MagmaLeft if side == "L" else ma.MagmaRight,
                                          ma.MagmaUpper if uplo == "U" else ma.MagmaLower,
                                          ma.MagmaNoTrans if trans == "N" else ma.MagmaTrans, ma.MagmaNonUnit, m, n, 1.0,
                                          dA.ptr, dA.ld, dB.ptr, dB.ld, count, queue.handle)
        X = dB.numpy()
        for s in range(4):
            want = oracle.dtrsm(side.encode(), uplo.encode(), trans.encode(), b"N", m, n, 1.0, F[s], B[s])
            assert same(X[s], want), (order, s)
            assert np.array_equal(X[s::4], np.broadcast_to(X[s], X[s::4].shape)), (order, s)


@pytest.mark.parametrize("count", [5, 4100])
@pytest.mark.parametrize("n,nrhs", [(1, 16), (1, 33), (2, 8), (2, 9), (2, 16), (2, 17), (4, 4), (4, 8), (4, 9), (5, 1), (8, 4),
                                    (8, 5), (9, 1)])
def test_tiny_solves(queue, oracle, count, n, nrhs):
    """Either side of the lines between the tiniest systems' kernel and the
    sweeps: getrs bitwise the oracle's, its transpose and potrs by the residual."""
    import magma_amd as ma
    import torch
    rng = np.random.default_rng(100 * n + nrhs)
    LU, ipiv = factor_batch(rng, 5, n)
    B = rng.uniform(-1, 1, (5, nrhs, n))
    many = lambda a: np.tile(a, (-(-count // 5),) + (1,) * (a.ndim - 1))[:count]      # noqa: E731
    ip = ma.IntBatch(count, n)
    ip.t.copy_(torch.from_numpy(many(ipiv)))
    print(f"tiny solves n={n} nrhs={nrhs} count={count}", flush=True)
    for op in ("N", "T", "potrs"):
        dA, dB = device(many(LU), n + 1), device(many(B), n + 2)
        if op == "potrs":
            assert ma.dpotrs_batched(dA, dB, queue, uplo=ma.MagmaLower) == 0
        else:
            assert ma.dgetrs_batched(dA, ip, dB, queue, trans=ma.MagmaNoTrans if op == "N" else ma.MagmaTrans) == 0
        X = dB.numpy()
        assert bool(dB.t[:, :, n:].isnan().all())
        for s in range(5):
            assert np.array_equal(X[s::5], np.broadcast_to(X[s], X[s::5].shape)), (op, s)
            L = np.tril(LU[s].T, -1) + np.eye(n)
            A = L @ np.triu(LU[s].T)                # rows in pivot order
            for k in reversed(range(n)):
                p = ipiv[s][k] - 1
                A[[k, p]] = A[[p, k]]
            if op == "N":
                assert same(X[s], oracle.dgetrs(LU[s], ipiv[s], B[s])), s
            elif op == "T":
                assert oracle.solve_error(A, X[s], B[s]) < 30, s
            else:
                C = np.tril(LU[s].T)
                assert oracle.solve_error(C @ C.T, X[s], B[s]) < 30, s


@pytest.mark.parametrize("n", [1, 2, 4, 5])
def test_getri_tiny(queue, oracle, n):
    """Above 4096 matrices of order up to 4: bitwise the oracle's dgetrs on the
    identity, info of a singular one."""
    import magma_amd as ma
    import torch
    rng = np.random.default_rng(n)
    count = 4101
    LU, ipiv = factor_batch(rng, 3, n)
    LU[1][n // 2, n // 2] = 0.0
    dA, dI = device(np.tile(LU, (count // 3, 1, 1)), n + 1), ma.DeviceBatch(np.full((count, n, n), 7.0), ld=n + 2)
    ip = ma.IntBatch(count, n)
    ip.t.copy_(torch.from_numpy(np.tile(ipiv, (count // 3, 1))))
    info = torch.full((count,), -1, dtype=torch.int32, device="cuda")
    print(f"getri tiny n={n}", flush=True)
    assert ma.load().magma_dgetri_outofplace_batched(n, dA.ptr, dA.ld, ip.ptr, dI.ptr, dI.ld, info.data_ptr(), count,
                                                     queue.handle) == 0
    X = dI.numpy()
    for s in range(3):
        assert same(X[s], oracle.dgetrs(LU[s], ipiv[s], np.eye(n))), s
        assert same(X[s::3], np.broadcast_to(X[s], X[s::3].shape)), s
    assert info.cpu().numpy().reshape(-1, 3).tolist() == [[0, n // 2 + 1, 0]] * (count // 3)
