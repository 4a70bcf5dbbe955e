"""GPU parity: the f32 product of up to 1024 rows (sgemm_rows_kernel of csrc/sgemm.hip) at the edges of its 16-row and
64-column tiles, of its 16-k steps and of its K splits, against float64. A sum of K fp32 products is off by at most
(K + 8) 2^-24 of the sum of its terms' magnitudes, whatever its order; the epilogue adds two roundings."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K", [(1, 1, 16), (2, 3, 17), (5, 70, 31), (16, 64, 128), (17, 65, 129), (33, 4, 200), (48, 257, 64), (64, 896, 4864),
                                   (65, 100, 1000), (127, 63, 16), (129, 130, 97), (200, 1153, 901), (333, 640, 896), (1000, 61, 65),
                                   (33, 16500, 16), (33, 16320, 16), (100, 25003, 20), (127, 40001, 33), (64, 70000, 47), (17, 33100, 16),
                                   (208, 5518, 296), (864, 4021, 308), (153, 17729, 245)])
def test_edges(lib, orc, M, N, K, tb):
    print("case sgemm rows", M, N, K, tb, flush=True)
    A, B = orc.normal(M * K, 61).reshape(M, K), orc.normal(N * K, 62).reshape((N, K) if tb else (K, N))
    Bd = (B.T if tb else B).astype(np.float64)
    want, mag = A.astype(np.float64) @ Bd, np.abs(A).astype(np.float64) @ np.abs(Bd)
    da, db, out = lib.to_device(A), lib.to_device(B), lib.to_device(np.full((M + 1, N), np.nan, np.float32))
    for scale, offset in ((1.0, 0.0), (-0.75, 2.0)):
        lib.gemm(da, K, 0, db, K if tb else N, tb, out, M, N, K, scale, offset)
        got = out.numpy()
        assert np.all(np.abs(got[:M] - (want * scale + offset)) <= (K + 8) * 2.0 ** -24 * mag * abs(scale) + 2.0 ** -22 * (np.abs(want * scale) + abs(offset)))
        assert np.isnan(got[M]).all()              # nothing past the result
    for b in (da, db, out):
        b.free()


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K", [(16, 70, 2100), (30, 131, 1300), (45, 67, 1607), (64, 129, 2049), (100, 65, 1500)])
def test_recorded_without_scratch(fresh_lib, recorded, orc, M, N, K, tb):
    """Where the parts of a split K have no room a block takes all of it: 10 to 17 steps to a wavefront, whose three or four
    slots of registers are filled several times, for one to four row tiles."""
    print("case sgemm rows recorded", M, N, K, tb, flush=True)
    A, B = orc.normal(M * K, 66).reshape(M, K), orc.normal(N * K, 67).reshape((N, K) if tb else (K, N))
    Bd = (B.T if tb else B).astype(np.float64)
    want, slack = A.astype(np.float64) @ Bd, (K + 8) * 2.0 ** -24 * (np.abs(A).astype(np.float64) @ np.abs(Bd))
    da, db, out = fresh_lib.to_device(A), fresh_lib.to_device(B), fresh_lib.empty((M, N))
    call = lambda m, n, k: fresh_lib.gemm(da, K, 0, db, K if tb else N, tb, out, m, n, k)
    call(1, 1, 16)                                 # (the first launch of a library loads its kernels)
    for got in recorded(lambda: call(M, N, K), out):
        assert np.all(np.abs(got - want) <= slack)
    before = fresh_lib.alloc_calls()
    call(M, N, K)                                  # with scratch to be had: in parts
    assert fresh_lib.alloc_calls() > before and np.all(np.abs(out.numpy() - want) <= slack)
    for b in (da, db, out):
        b.free()


@pytest.mark.parametrize("M,N,K", [(20, 130, 37), (70, 90, 700)])
def test_infinities_and_nan_stay_where_they_are(lib, orc, M, N, K):
    """A row with an infinity gives infinities of the sign of the column's weight, one with a NaN gives NaN, a zero
    against an infinity NaN; every other row is untouched by them (rows and k past the edges are read clamped)."""
    A, B = orc.normal(M * K, 63).reshape(M, K), orc.normal(N * K, 64).reshape(K, N)
    A[M - 1, K - 1], A[3, 5] = np.inf, np.nan
    B[K - 1, 7] = 0.0
    da, db, out = lib.to_device(A), lib.to_device(B), lib.empty((M, N))
    lib.gemm(da, K, 0, db, N, 0, out, M, N, K)
    got, rest = out.numpy(), [r for r in range(M) if r not in (3, M - 1)]
    assert np.isnan(got[3]).all() and np.isnan(got[M - 1, 7])
    other = [c for c in range(N) if c != 7]
    assert np.array_equal(got[M - 1, other], np.where(B[K - 1, other] > 0, np.inf, -np.inf))
    want = A[rest].astype(np.float64) @ B.astype(np.float64)
    assert np.all(np.abs(got[rest] - want) <= (K + 8) * 2.0 ** -24 * (np.abs(A[rest]).astype(np.float64) @ np.abs(B).astype(np.float64)))
    for b in (da, db, out):
        b.free()


def test_strided_views_and_byte_offsets(lib, orc):
    """Operands inside larger buffers at offsets that are not multiples of 16 bytes; integers come out exact."""
    rng = np.random.default_rng(65)
    M, N, K, la, lb = 37, 75, 83, 91, 79
    A, B = rng.integers(-50, 50, (M + 2, la)).astype(np.float32), rng.integers(-50, 50, (K + 1, lb)).astype(np.float32)
    da, db, out = lib.to_device(A), lib.to_device(B), lib.empty(M * N + 3)
    lib._chk(lib.c.tlhip_gemm(da.ptr, (la + 3) * 4, la, 0, db.ptr, 1 * 4, lb, 0, out.ptr, 3 * 4, M, N, K, 1.0, 0.0))
    want = A[1:M + 1, 3:3 + K].astype(np.float64) @ B[:K, 1:1 + N].astype(np.float64)
    assert np.array_equal(out.numpy()[3:].reshape(M, N).astype(np.float64), want)
    for b in (da, db, out):
        b.free()


def test_more_columns_than_a_grid_of_its_blocks_counts(lib, orc):
    """2^29 columns and a few: one row of B is read for all of them (a row stride of zero), so only the result is large."""
    N, K = (1 << 29) + 70, 16
    a, b = np.arange(1, K + 1, dtype=np.float32), np.arange(K, dtype=np.float32) - 5
    da, db, out = lib.to_device(a), lib.to_device(b), lib.empty_bytes(N * 4)
    lib.gemm(da, K, 0, db, 0, 1, out, 1, N, K)
    for first in (0, (1 << 28) - 7, N - 1000):
        got = np.empty(1000, np.float32)
        lib._chk(lib.c.tlhip_memcpy_d2h(got.ctypes.data, out.ptr + first * 4, got.nbytes))
        assert np.all(got == a @ b), first
    for x in (da, db, out):
        x.free()
