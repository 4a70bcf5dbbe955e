"""GPU parity: int4 products of more than 64 rows (csrc/gemm_q4.hip) at the edges of their 64-row and 256-column tiles, of
their units of four groups (K not a multiple of 128 too) and of their K splits, against float64.

Activations enter as two f16 terms of a row scaled by a power of two: 2^-24 of each product's magnitude (the cases' rows
hold no element 2^24 below their largest); the sums are fp32, 32 products inside two instructions per term, then one
addition per group and one per part."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(lib, orc, M, rows, K, seed):
    A = orc.normal(M * K, seed).reshape(M, K)
    A = np.where(np.abs(A) < 1e-4, np.float32(1e-4), A).astype(np.float32)
    rng = np.random.default_rng(seed)
    packed = rng.integers(0, 256, (rows, K // 2), dtype=np.uint8)
    scales = rng.uniform(0.002, 0.006, (rows, K // 32)).astype(np.float32)
    nib = np.stack([packed & 15, packed >> 4], -1).reshape(rows, K // 32, 32).astype(np.float64) - 8
    W, A64 = (nib * scales[:, :, None]).reshape(rows, K), A.astype(np.float64)
    slack = (K / 32 + 100) * 2.0 ** -24 * (np.abs(A64) @ np.abs(W).T)
    return lib.to_device(A), lib.to_device(np.concatenate([packed.ravel(), scales.ravel().view(np.uint8)])), A64 @ W.T, slack


@pytest.mark.parametrize("M,N,K", [(65, 2048, 32), (129, 2049, 160), (200, 257, 896), (192, 2304, 128), (301, 2500, 1056), (320, 4608, 3584),
                                   (512, 3584, 1024), (193, 70000, 256), (1000, 2300, 384),
                                   (847, 9344, 256)])
def test_plain_and_parts(lib, orc, M, N, K):
    print("case gemm_q4", M, N, K, flush=True)
    da, dw, want, slack = _case(lib, orc, M, N, K, 81)
    out = lib.to_device(np.full((M, N), np.nan, np.float32))
    parts = lib.to_device(np.full((4, M, N), np.nan, np.float32))
    lib.gemm_q4_nt(da, dw, out, M, N, K)
    n = lib.gemm_q4_nt_parts(da, dw, parts, M, N, K)
    assert 1 <= n <= 4
    assert np.all(np.abs(out.numpy() - want) <= slack)
    got = parts.numpy()
    assert np.all(np.abs(got[:n].astype(np.float64).sum(0) - want) <= slack)
    assert np.isnan(got[n:]).all()
    for b in (da, dw, out, parts):
        b.free()


@pytest.mark.parametrize("M,ff,K", [(66, 1024, 32), (129, 1100, 160), (301, 4864, 896), (512, 1030, 384), (200, 18944, 128),
                                    (731, 2304, 416), (727, 1501, 416)])
def test_gated(lib, orc, M, ff, K):
    print("case gemm_q4 gated", M, ff, K, flush=True)
    da, dw, p, s = _case(lib, orc, M, 2 * ff, K, 83)
    g, u, sg, su = p[:, :ff], p[:, ff:], s[:, :ff], s[:, ff:]
    act, out = g / (1 + np.exp(-g)), lib.to_device(np.full((M, ff), np.nan, np.float32))
    lib.gemm_q4_nt_swiglu(da, dw, out, M, ff, K)
    # the slope of x sigmoid(x) is below 1.1; the gate itself costs a few roundings
    assert np.all(np.abs(out.numpy() - act * u) <= 1.1 * sg * (np.abs(u) + su) + np.abs(act) * su + 1e-6 * np.abs(act * u))
    for b in (da, dw, out):
        b.free()


@pytest.mark.parametrize("M,K", [(65, 2016), (65, 2080), (65, 4064), (65, 4128), (65, 8160), (65, 8224), (65, 20448), (65, 20512), (65, 32736),
                                 (65, 32800), (129, 2048), (129, 4096), (129, 20480), (129, 32768)])
def test_rows_at_the_limits_of_the_images_kernels(lib, orc, M, K):
    """A row's image is cut by threads that hold the whole row: one to sixteen runs of eight k each, to 2048, 4096, 8192, 20480 and
    32768 k. Longer rows are multiplied without images."""
    N = 2048
    print("case gemm_q4 limits", M, N, K, flush=True)
    da, dw, want, slack = _case(lib, orc, M, N, K, 85)
    out = lib.to_device(np.full((M, N), np.nan, np.float32))
    lib.gemm_q4_nt(da, dw, out, M, N, K)
    assert np.all(np.abs(out.numpy() - want) <= slack)
    for b in (da, dw, out):
        b.free()


def test_infinities_and_nan_stay_in_their_rows(lib, orc):
    M, N, K = 301, 2049, 896
    print("case gemm_q4 not finite", M, N, K, flush=True)
    da, dw, _, _ = _case(lib, orc, M, N, K, 87)
    out, A = lib.empty((M, N)), da.numpy()
    lib.gemm_q4_nt(da, dw, out, M, N, K)
    clean = out.numpy()
    A[3, 5], A[200, K - 1] = np.inf, np.nan
    lib.gemm_q4_nt(da.upload(A), dw, out, M, N, K)
    got, rest = out.numpy(), [r for r in range(M) if r not in (3, 200)]
    assert np.isnan(got[[3, 200]]).all() and np.array_equal(got[rest], clean[rest])
    for b in (da, dw, out):
        b.free()


@pytest.mark.parametrize("M,N,K", [(301, 2049, 928), (301, 2049, 960), (65, 2049, 2080), (512, 3584, 992), (129, 2049, 160)])
def test_infinities_and_nan_ahead_of_a_broken_unit(lib, orc, M, N, K):
    """K % 128 of 32, 64 and 96: the last unit of four groups lacks some, and what stands in for them must not carry the last group's
    elements of rows 48 .. 63 of a block to the other rows: the others are the clean product's, bit for bit."""
    print("case gemm_q4 not finite, broken unit", M, N, K, flush=True)
    da, dw, _, _ = _case(lib, orc, M, N, K, 93)
    out, act, A = lib.empty((M, N)), lib.empty((M, N // 2)), da.numpy()
    forms = ((out, lambda: lib.gemm_q4_nt(da, dw, out, M, N, K)), (act, lambda: lib.gemm_q4_nt_swiglu(da, dw, act, M, N // 2, K)))
    clean = []
    for o, call in forms if N % 2 == 0 else forms[:1]:
        call()
        clean.append(o.numpy())
    bad = [r for r in (48, 63, 126, M - 2) if r < M]
    A[bad[0], K - 1], A[bad[1], K - 9] = np.inf, np.nan
    for r in bad[2:]:
        A[r, K - 32] = -np.inf
    da.upload(A)
    rest = [r for r in range(M) if r not in bad]
    for (o, call), c in zip(forms, clean):
        call()
        got = o.numpy()
        assert np.array_equal(got[rest], c[rest]), [r for r in rest if not np.array_equal(got[r], c[r])]
        assert not np.isfinite(got[bad]).any()
    for b in (da, dw, out, act):
        b.free()


def test_recorded_without_room_for_the_images(fresh_lib, recorded, orc):
    """The images of 200 rows of 16384 take 16 MB; a recording that finds 8 MB multiplies without them."""
    M, N, K = 200, 2049, 16384
    print("case gemm_q4 recorded", M, N, K, flush=True)
    da, dw, want, slack = _case(fresh_lib, orc, M, N, K, 89)
    out = fresh_lib.empty((M, N))
    fresh_lib.gemm_q4_nt(da, dw, out, 65, 2048, 32)   # (scratch comes in 8 MB at least)
    for got in recorded(lambda: fresh_lib.gemm_q4_nt(da, dw, out, M, N, K), out):
        assert np.all(np.abs(got - want) <= slack)
    before = fresh_lib.alloc_calls()
    fresh_lib.gemm_q4_nt(da, dw, out, M, N, K)
    assert fresh_lib.alloc_calls() > before and np.all(np.abs(out.numpy() - want) <= slack)
    for b in (da, dw, out):
        b.free()


def test_recorded_without_room_for_parts(fresh_lib, recorded, orc):
    """359 rows of this weight are formed without images, in two parts of 31 MB; a recording with room for the images only (3 MB)
    takes those."""
    M, N, K = 359, 10880, 1792
    print("case gemm_q4 recorded parts", M, N, K, flush=True)
    da, dw, want, slack = _case(fresh_lib, orc, M, N, K, 91)
    out = fresh_lib.empty((M, N))
    fresh_lib.gemm_q4_nt(da, dw, out, 65, 2048, 32)   # (scratch comes in 8 MB at least)
    for got in recorded(lambda: fresh_lib.gemm_q4_nt(da, dw, out, M, N, K), out):
        assert np.all(np.abs(got - want) <= slack)
    for b in (da, dw, out):
        b.free()
