"""GPU parity: f32 products on the bf16 matrix pipe in three terms (sgemm_split_kernel of csrc/sgemm_split.hip) at the edges of its 32-row
and 128-column tiles, its 16-k steps and its K splits, and over the whole range of f32, where it hands a tile to the fp32 pipe, against
float64. A sum of K fp32 products is off by at most (K + 8) 2^-24 of the sum of its terms' magnitudes, whatever its order, and the terms
left out add up to 2^-24 of each; a product below the least normal number may be lost. That holds for any kernel and would hide a term
gone missing, so the error over a whole result is compared with the fp32 pipe's too. The sizes are such that the estimates choose it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TINY = 2.0 ** -126


def _run(lib, A, B, tb, scale=1.0, offset=0.0):
    (M, K), N = A.shape, B.shape[0] if tb else B.shape[1]
    da, db, out = lib.to_device(A), lib.to_device(B), lib.to_device(np.full((M + 1, N), np.nan, np.float32))
    lib.gemm(da, K, 0, db, K if tb else N, tb, out, M, N, K, scale, offset)
    got = out.numpy()
    assert np.isnan(got[M]).all()                  # nothing past the result
    for b in (da, db, out):
        b.free()
    return got[:M]


def _near(got, A, B, tb, scale=1.0, offset=0.0, rows=slice(None)):
    A64, B64 = A[rows].astype(np.float64), (B.T if tb else B).astype(np.float64)
    K = A.shape[1]
    slack = (K + 9) * 2.0 ** -24 * (np.abs(A64) @ np.abs(B64)) * abs(scale) + K * TINY
    if (scale, offset) != (1.0, 0.0):
        slack += 2.0 ** -22 * (np.abs(A64 @ B64 * scale) + abs(offset))
    assert np.all(np.abs(got[rows] - (A64 @ B64 * scale + offset)) <= slack)


# one row tile and two, a last tile of one row and of all but one; 128 columns and one more; whole steps, one k more, one short; splits
@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K", [(97, 5000, 1024), (128, 4097, 1025), (97, 9000, 1039), (193, 4864, 896), (700, 129, 4000), (320, 1152, 2049),
                                   (333, 4861, 901), (512, 2048, 1024), (600, 128, 4864), (1024, 1279, 530), (64, 12000, 1100), (500, 896, 4864)])
def test_edges(lib, orc, M, N, K, tb):
    print("case sgemm split", M, N, K, tb, flush=True)
    A, B = orc.normal(M * K, 71).reshape(M, K), orc.normal(N * K, 72).reshape((N, K) if tb else (K, N))
    for scale, offset in ((1.0, 0.0), (-0.75, 2.0)):
        _near(_run(lib, A, B, tb, scale, offset), A, B, tb, scale, offset)


@pytest.mark.parametrize("tb", [0, 1])
def test_any_magnitude(lib, orc, tb):
    """Rows from 2^-140 to 2^120 in one matrix, single elements far below or above their row, rows and columns of zeros."""
    M, N, K = 160, 4900, 900
    A, B = orc.normal(M * K, 73).reshape(M, K), orc.normal(N * K, 74).reshape((N, K) if tb else (K, N))
    A *= np.exp2(np.linspace(-140, 60, M)).astype(np.float32)[:, None]
    A[7] = 0
    A[100:140] = orc.normal(40 * K, 75).reshape(40, K)   # row tiles of ordinary numbers ...
    A[110, 3], A[111, 4] = 2.0 ** -149, 2.0 ** 126       # ... but for these
    A[112] *= 2.0 ** -60
    got = _run(lib, A, B, tb)
    _near(got, A, B, tb)
    assert np.all(got[7] == 0)
    B2 = B * np.float32(2.0 ** -70)                      # products below 2^-126 of ordinary rows
    _near(_run(lib, A, B2, tb), A, B2, tb)


@pytest.mark.parametrize("tb", [0, 1])
def test_infinities_and_nan_stay_where_they_are(lib, orc, tb):
    M, N, K = 200, 4864, 896
    A, B = orc.normal(M * K, 76).reshape(M, K), orc.normal(N * K, 77).reshape((N, K) if tb else (K, N))
    A[M - 1, K - 1], A[3, 5] = np.inf, np.nan
    Bk = B.T if tb else B                                # a view of what is uploaded
    Bk[K - 1, 7] = 0.0
    Bk[K - 1, 8:16] = 1.0                                # whose lower terms are zeros
    Bk[11, 300] = -np.inf
    got, rows = _run(lib, A, B, tb), [r for r in range(M) if r not in (3, M - 1)]
    assert np.isnan(got[3]).all() and np.isnan(got[M - 1, 7])
    other = [c for c in range(N) if c not in (7, 300)]
    assert np.array_equal(got[M - 1, other], np.where(Bk[K - 1, other] > 0, np.inf, -np.inf))
    assert np.array_equal(got[rows, 300], np.where(A[rows, 11] > 0, -np.inf, np.inf))
    Bf = B.copy()
    (Bf.T if tb else Bf)[11, 300] = 0
    keep = [c for c in range(N) if c != 300]
    A64, B64 = A[rows].astype(np.float64), (Bf.T if tb else Bf).astype(np.float64)
    assert np.all(np.abs(got[np.ix_(rows, keep)] - (A64 @ B64)[:, keep]) <= ((K + 9) * 2.0 ** -24 * (np.abs(A64) @ np.abs(B64)))[:, keep])


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K", [(193, 4865, 896), (333, 4861, 901), (700, 129, 4000), (500, 897, 4864)])
def test_one_writer_for_each_column(lib, orc, M, N, K, tb):
    """The last column tile is moved back to end with the matrix and reads columns that the one before it owns. A number that sends only
    one of the two to the fp32 pipe leaves the other's columns their bits."""
    print("case sgemm split overlap", M, N, K, tb, flush=True)
    A, B = orc.normal(M * K, 81).reshape(M, K), orc.normal(N * K, 82).reshape((N, K) if tb else (K, N))
    clean, first = _run(lib, A, B, tb), N // 128 * 128
    for column, kept in ((N - 1, slice(0, first)), (first - 128, slice(first, N))):
        for value in (2.0 ** -140, 2.0 ** 120):
            Bx = B.copy()
            (Bx.T if tb else Bx)[5, column] = value      # read by the last tile only, then by the one before it only
            got = [_run(lib, A, Bx, tb) for _ in range(3)]
            assert np.array_equal(got[0][:, kept], clean[:, kept]) and np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K", [(333, 4864, 896), (99, 4608, 3584), (500, 896, 4864), (700, 129, 4000), (320, 1152, 2049), (512, 2048, 1024)])
def test_no_further_off_than_the_fp32_pipe(lib, orc, M, N, K, tb):
    """The same numbers with A transposed go to the LDS-tiled fp32 kernel, which adds all of a block's K in one chain: 1.7 to 5.5 times this
    kernel's error in these shapes (2-norm). Without the third terms of one operand the result would be
    off by 2.4e-6, twice that kernel's error at its largest (1.1e-6)."""
    print("case sgemm split error", M, N, K, tb, flush=True)
    A, B = orc.normal(M * K, 85).reshape(M, K), orc.normal(N * K, 86).reshape((N, K) if tb else (K, N))
    want = A.astype(np.float64) @ (B.T if tb else B).astype(np.float64)
    err = lambda got: np.linalg.norm(got - want) / np.linalg.norm(want)
    da, db, out = lib.to_device(np.ascontiguousarray(A.T)), lib.to_device(B), lib.empty((M, N))
    lib.gemm(da, M, 1, db, K if tb else N, tb, out, M, N, K)
    fp32, here = err(out.numpy()), err(_run(lib, A, B, tb))
    assert here <= fp32, (here, fp32)
    for b in (da, db, out):
        b.free()


@pytest.mark.parametrize("tb", [0, 1])
def test_sums_of_one_product(lib, orc, tb):
    """Rows with a single element. Eight bits of it lose nothing, so that rows are selected and scaled by powers of two exactly. Of 24
    bits the two pairs left out are at most 2^-24 of the product, half a unit in the last place of a result just above a power of two and one of
    the largest, and the pipe's last addition is off by less than one: below 2 units (measured 1.43, and 0.5 on the fp32 pipe)."""
    M, N, K = 333, 4864, 896
    at, B = (np.arange(M) * 7) % K, orc.normal(N * K, 88).reshape((N, K) if tb else (K, N))
    Bk = B.T if tb else B
    for values in (np.ones(M), np.exp2(np.arange(M) % 9 - 4), 1 + np.arange(M) % 256):
        A = np.zeros((M, K), np.float32)
        A[np.arange(M), at] = values
        got, want = _run(lib, A, B, tb), Bk[at].astype(np.float64) * values[:, None]
        if values.max() < 100:
            assert np.array_equal(got, want.astype(np.float32))
        else:                                            # (32 bits: rounded, by the last addition)
            assert np.all(np.abs(got - want) < np.spacing(np.abs(want).astype(np.float32)))
    A[np.arange(M), at] = orc.normal(M, 89)
    want = Bk[at].astype(np.float64) * A[np.arange(M), at].astype(np.float64)[:, None]
    assert np.all(np.abs(_run(lib, A, B, tb) - want) < 2 * np.spacing(np.abs(want).astype(np.float32)))


def test_whole_numbers_are_exact(lib):
    """Products that fit 24 bits lose no term: 10 bits by 6, 15 by 2 and the other way round, each sum below 2^24."""
    g = np.random.default_rng(78)
    for bits_a, bits_b in ((9, 5), (14, 1), (1, 14)):
        A = g.integers(-(1 << bits_a), (1 << bits_a) + 1, (160, 900)).astype(np.float32)
        B = g.integers(-(1 << bits_b), (1 << bits_b) + 1, (900, 4900)).astype(np.float32)
        assert np.array_equal(_run(lib, A, B, 0).astype(np.float64), A.astype(np.float64) @ B.astype(np.float64))


@pytest.mark.parametrize("M,N,K", [(333, 896, 4864), (130, 3584, 3584)])
def test_recorded(fresh_lib, recorded, orc, M, N, K):
    """Recorded where the parts have no room (another kernel takes it), and eagerly, where they have."""
    A, B = orc.normal(M * K, 79).reshape(M, K), orc.normal(N * K, 80).reshape(K, N)
    want = A.astype(np.float64) @ B.astype(np.float64)
    slack = (K + 9) * 2.0 ** -24 * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64))
    da, db, out = fresh_lib.to_device(A), fresh_lib.to_device(B), fresh_lib.empty((M, N))
    call = lambda: fresh_lib.gemm(da, K, 0, db, N, 0, out, M, N, K)
    fresh_lib.gemm(da, 16, 0, db, 1, 0, out, 1, 1, 16)     # (the first launch of a library loads its kernels)
    for got in recorded(call, out):
        assert np.all(np.abs(got - want) <= slack)
    call()
    eager = out.numpy().copy()
    assert np.all(np.abs(eager - want) <= slack)
    fresh_lib.graph_begin()                                # with room now
    call()
    g = fresh_lib.graph_end()
    for _ in range(3):
        out.upload(np.full((M, N), np.nan, np.float32))
        fresh_lib.graph_launch(g)
        fresh_lib.sync()
        assert np.array_equal(out.numpy(), eager)
    fresh_lib.graph_destroy(g)
    for b in (da, db, out):
        b.free()
