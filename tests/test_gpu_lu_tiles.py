"""LU for 64 < max(m, n) <= 512: orders and shapes at the edges of the 32-column
blocks, the 16-row tiles and the three kernels' ranges, and matrices that leave
the fast path (ties, NaN, infinities, overflow, pivots below DBL_MIN) at
different depths.  Factors, pivots and info are the oracle's bits: every entry
gets the same fused multiply-adds in the same order, so the tolerance is zero."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(65, 65, 65), (97, 128, 99), (128, 33, 128), (129, 129, 131), (159, 161, 159), (161, 159, 161),
          (255, 256, 255), (256, 40, 256), (40, 256, 48), (257, 257, 257), (300, 511, 301), (512, 70, 512),
          (70, 512, 70), (497, 497, 500), (512, 512, 512)]


def same(a, b):
    return a.shape == b.shape and bool(np.all((a == b) | (np.isnan(a) & np.isnan(b))))


@pytest.mark.parametrize("m,n,ld", SHAPES)
def test_getrf_shapes(queue, oracle, m, n, ld):
    import magma_amd as ma
    rng = np.random.default_rng(1000 * m + n)
    A = rng.uniform(-1, 1, (3, n, m))
    print(f"getrf m={m} n={n} ld={ld}", flush=True)
    dA = ma.DeviceBatch(A, ld=ld)
    ret, ipiv, info = ma.dgetrf_batched(dA, queue, m=m, n=n)
    assert ret == 0
    got, ip, inf = dA.numpy(), ipiv.numpy(), info.cpu().numpy()
    for s in range(3):
        LUo, ipo, info_o = oracle.dgetrf(A[s], m=m, n=n)
        assert inf[s] == info_o and np.array_equal(ip[s], ipo) and same(got[s], LUo), s


@pytest.mark.parametrize("n", [130, 257])
def test_getrf_special(queue, oracle, n):
    import magma_amd as ma
    rng = np.random.default_rng(n)
    mats = []
    for t in range(7):
        A = rng.integers(-2, 3, size=(n, n)).astype(float)      # ties in the pivot search
        if t == 1:
            A[:, n // 2] = 0.0
        if t == 2:
            A[n - 3] = A[5]
        if t == 3:
            A[n // 3, (2 * n) // 3] = np.nan
        if t == 4:
            A[7, n - 30], A[n - 9, 40] = np.inf, -np.inf
        if t == 5:
            A *= 1e300                                          # overflows during the updates
        if t == 6:
            A[:, 33] *= 1e-310                                  # pivots below DBL_MIN
            A[:, n - 2] *= 1e-312
        mats.append(A.T.copy())
    mats.append(np.zeros((n, n)))
    mats.append(np.eye(n)[::-1].T.copy())
    A = np.stack(mats)
    print(f"getrf special n={n}", flush=True)
    dA = ma.DeviceBatch(A)
    ret, ipiv, info = ma.dgetrf_batched(dA, queue)
    assert ret == 0
    LUo, ipo, info_o = oracle.batch_dgetrf(A)
    assert np.array_equal(info.cpu().numpy(), info_o)
    assert np.array_equal(ipiv.numpy(), ipo)
    assert same(dA.numpy(), LUo)


@pytest.mark.parametrize("nocheck", [False, True])
def test_getrf_vbatched_empty(queue, oracle, nocheck):
    """Matrices without rows or columns, with null pointers, in every size class
    of the kernel beside ordinary ones: info 0, nothing read, the others as ever."""
    import magma_amd as ma
    rng = np.random.default_rng(11)
    shapes = [(0, 100), (100, 0), (70, 66), (0, 200), (256, 0), (130, 129), (300, 0), (0, 512), (257, 40)]
    V = ma.VarBatch([rng.uniform(-1, 1, (n, m)) for m, n in shapes])
    for i, (m, n) in enumerate(shapes):
        if m == 0 or n == 0:
            V.ptrs[i] = 0
    ipiv = ma.VarInts([max(1, min(s)) for s in shapes])
    info = ma.dev_ints(np.full(len(shapes), -1))
    print(f"getrf_vbatched with empty matrices nocheck={nocheck}", flush=True)
    before = V.matrices()
    L = ma.load()
    if nocheck:
        ret = L.magma_dgetrf_vbatched_max_nocheck(V.d_rows.data_ptr(), V.d_cols.data_ptr(), 512, V.ptr,
                                                  V.d_ld.data_ptr(), ipiv.ptr, info.data_ptr(), V.count, queue.handle)
        queue.sync()
    else:
        ret = L.magma_dgetrf_vbatched(V.d_rows.data_ptr(), V.d_cols.data_ptr(), V.ptr, V.d_ld.data_ptr(), ipiv.ptr,
                                      info.data_ptr(), V.count, queue.handle)
    assert ret == 0
    assert info.cpu().numpy()[: V.count].tolist() == [0] * V.count
    got = V.matrices()
    for i, (m, n) in enumerate(shapes):
        if m and n:
            LUo, ipo, _ = oracle.dgetrf(before[i], m=m, n=n)
            assert np.array_equal(ipiv.numpy(i, min(m, n)), ipo) and same(got[i], LUo), i


# either side of the lines between the kernels: rows 128 / 256, a side of 16
NARROW = [(8, 65), (65, 8), (16, 100), (17, 100), (16, 512), (17, 512), (128, 16), (129, 16), (129, 17), (300, 16),
          (300, 17), (512, 1), (1, 512), (100, 512), (128, 400), (129, 400), (64, 300)]


@pytest.mark.parametrize("m,n", NARROW)
def test_getrf_wide_and_narrow(queue, oracle, m, n):
    import magma_amd as ma
    rng = np.random.default_rng(1000 * m + n)
    A = rng.uniform(-1, 1, (3, n, m))
    A[2] = rng.integers(-2, 3, size=(n, m))          # ties
    print(f"getrf m={m} n={n}", flush=True)
    dA = ma.DeviceBatch(A, ld=m + 1)
    ret, ipiv, info = ma.dgetrf_batched(dA, queue, m=m, n=n)
    assert ret == 0
    got, ip, inf = dA.numpy(), ipiv.numpy(), info.cpu().numpy()
    for s in range(3):
        LUo, ipo, info_o = oracle.dgetrf(A[s], m=m, n=n)
        assert inf[s] == info_o and np.array_equal(ip[s], ipo) and same(got[s], LUo), s


@pytest.mark.parametrize("nocheck", [False, True])
def test_getrf_vbatched_wide_and_narrow(queue, oracle, nocheck):
    """The same shapes in one variable-size call, where wide matrices go by their rows."""
    import magma_amd as ma
    rng = np.random.default_rng(12)
    shapes = NARROW + [(70, 600), (600, 70), (64, 64), (60, 65)]
    mats = [rng.uniform(-1, 1, (n, m)) for m, n in shapes]
    V = ma.VarBatch(mats)
    ipiv = ma.VarInts([min(s) for s in shapes])
    info = ma.dev_ints(np.full(len(shapes), -1))
    print(f"getrf_vbatched wide and narrow nocheck={nocheck}", flush=True)
    L = ma.load()
    if nocheck:
        ret = L.magma_dgetrf_vbatched_max_nocheck(V.d_rows.data_ptr(), V.d_cols.data_ptr(), 600, V.ptr,
                                                  V.d_ld.data_ptr(), ipiv.ptr, info.data_ptr(), V.count, queue.handle)
        queue.sync()
    else:
        ret = L.magma_dgetrf_vbatched(V.d_rows.data_ptr(), V.d_cols.data_ptr(), V.ptr, V.d_ld.data_ptr(), ipiv.ptr,
                                      info.data_ptr(), V.count, queue.handle)
    assert ret == 0
    assert info.cpu().numpy()[: V.count].tolist() == [0] * V.count
    got = V.matrices()
    for i, (m, n) in enumerate(shapes):
        LUo, ipo, _ = oracle.dgetrf(mats[i], m=m, n=n)
        assert np.array_equal(ipiv.numpy(i, min(m, n)), ipo) and same(got[i], LUo), (m, n)


@pytest.mark.parametrize("m,n", [(33, 160), (70, 200), (128, 300), (200, 420)])
def test_getrf_special_wide(queue, oracle, m, n):
    """Block columns past the last pivot, which go to the rows' final places at
    once: after a fallback in the square part, in one of their own, and with
    an overflow in their updates."""
    import magma_amd as ma
    rng = np.random.default_rng(m)
    A = rng.uniform(-1, 1, (5, n, m))
    A[1][m // 2, m // 3] = np.nan                    # storage (column, row)
    A[2][m + 40, 7], A[2][n - 1, m - 1] = np.inf, np.nan
    A[3] = rng.integers(-2, 3, size=(n, m)) * 1e300
    A[4][:, 5] = 0.0                                 # a zero row: zeros in U under the fallback's skip
    A[4][n - 3, 2] = np.inf
    print(f"getrf wide m={m} n={n}", flush=True)
    dA = ma.DeviceBatch(A, ld=m + 1)
    ret, ipiv, info = ma.dgetrf_batched(dA, queue, m=m, n=n)
    assert ret == 0
    got, ip, inf = dA.numpy(), ipiv.numpy(), info.cpu().numpy()
    for s in range(5):
        LUo, ipo, info_o = oracle.dgetrf(A[s], m=m, n=n)
        assert inf[s] == info_o and np.array_equal(ip[s], ipo) and same(got[s], LUo), s
