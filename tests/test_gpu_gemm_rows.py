"""GPU parity: the products of a few rows (csrc/gemm_rows.hip) at the edges of their tiles: rows around the 16-row
tiles and the blocks of up to five of them, columns that fill no tile, K of one step, of fewer steps than wavefronts and
of many steps to a wavefront, both weight formats, plain, gated and left as K-split parts.

Every product is compared with float64. A sum of n fp32 additions is off by at most n 2^-24 of the sum of its terms'
magnitudes; here n is three terms per 32-k step of a wavefront's chain, the 32 products inside an instruction and the
eight wavefronts' sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 16, 128), (2, 33, 128), (5, 200, 256), (16, 896, 896), (17, 130, 128), (37, 1152, 896), (64, 64, 3584),
          (65, 100, 128), (77, 896, 4864), (80, 36, 2048), (81, 260, 384), (97, 128, 896), (128, 72, 640),
          (9, 18500, 128), (16, 18300, 128), (60, 33000, 128),
          # above 128 rows (bf16), few rows and columns of a long K; 1025 rows run in the tiles
          (129, 100, 896), (161, 48, 384), (255, 1200, 512), (256, 33, 4096), (7, 16, 12288), (11, 40, 9216),
          (257, 1152, 896), (336, 100, 2560), (401, 36, 4864), (1024, 48, 384), (1025, 40, 128),
          (129, 999, 8192), (200, 1151, 4864)]     # K cannot be split


def _weights(orc, fmt, N, K, seed):
    """(device bytes, float64 values) of an [N, K] weight."""
    if fmt == "bf16":
        w = orc.to_bf16(orc.normal(N * K, seed, std=0.02)).reshape(N, K)
        return w, orc.bf16_widen(w).reshape(N, K).astype(np.float64)
    rng = np.random.default_rng(seed)
    packed = rng.integers(0, 256, (N, K // 2), dtype=np.uint8)
    scales = rng.uniform(0.002, 0.006, (N, K // 32)).astype(np.float32)
    nib = np.stack([packed & 15, packed >> 4], -1).reshape(N, K // 32, 32).astype(np.float64) - 8
    return np.concatenate([packed.ravel(), scales.ravel().view(np.uint8)]), (nib * scales[:, :, None]).reshape(N, K)


def _slack(A, W, K):
    return (3 * K / 32 + 40) * 2.0 ** -24 * (np.abs(A) @ np.abs(W).T)


@pytest.mark.parametrize("fmt", ["bf16", "q4"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_plain_and_parts(lib, orc, fmt, M, N, K):
    print("case gemm_rows", fmt, M, N, K, flush=True)
    A = orc.normal(M * K, 21).reshape(M, K)
    w, W = _weights(orc, fmt, N, K, 22)
    want, slack = A.astype(np.float64) @ W.T, _slack(A.astype(np.float64), W, K)
    da, dw = lib.to_device(A), lib.to_device(w)
    out, parts = lib.to_device(np.full((M, N), np.nan, np.float32)), lib.to_device(np.full((16, M, N), np.nan, np.float32))
    if fmt == "bf16":
        lib.gemm_bf16_nt(da, dw, out, M, N, K)
        n = lib.gemm_bf16_nt_parts(da, dw, parts, M, N, K)
    else:
        lib.gemm_q4_nt(da, dw, out, M, N, K)
        n = lib.gemm_q4_nt_parts(da, dw, parts, M, N, K)
    assert 1 <= n <= 16
    assert np.all(np.abs(out.numpy() - want) <= slack)
    got = parts.numpy()
    assert np.all(np.abs(got[:n].astype(np.float64).sum(0) - want) <= slack)
    assert np.isnan(got[n:]).all()                 # nothing written past the parts
    for b in (da, dw, out, parts):
        b.free()


@pytest.mark.parametrize("fmt", ["bf16", "q4"])
@pytest.mark.parametrize("M,N,K", [(50, 890, 4864), (90, 17, 8192), (200, 890, 4864), (500, 300, 2048), (130, 3590, 1024), (300, 1000, 8192)])
def test_parts_and_tiles_in_runs(lib, orc, fmt, M, N, K):
    """Tiles that are no multiple of 8, fewer than 8 and several row blocks, times K-split parts: every part of every tile once."""
    test_plain_and_parts(lib, orc, fmt, M, N, K)


@pytest.mark.parametrize("fmt", ["bf16", "q4"])
@pytest.mark.parametrize("M,ff,K", [(1, 8, 128), (5, 4864, 896), (16, 100, 128), (33, 31, 256), (77, 4864, 896), (81, 200, 384), (128, 17, 128), (300, 200, 896), (16, 40, 4864), (40, 72, 4864),
                                    (150, 4864, 896), (200, 25, 1024)])
def test_gated(lib, orc, fmt, M, ff, K):
    print("case gemm_rows gated", fmt, M, ff, K, flush=True)
    A = orc.normal(M * K, 23).reshape(M, K)
    w, W = _weights(orc, fmt, 2 * ff, K, 24)
    p, s = A.astype(np.float64) @ W.T, _slack(A.astype(np.float64), W, K)
    g, u, sg, su = p[:, :ff], p[:, ff:], s[:, :ff], s[:, ff:]
    act = g / (1 + np.exp(-g))
    da, dw, out = lib.to_device(A), lib.to_device(w), lib.to_device(np.full((M, ff), np.nan, np.float32))
    (lib.gemm_bf16_nt_swiglu if fmt == "bf16" else lib.gemm_q4_nt_swiglu)(da, dw, out, M, ff, K)
    # the slope of x sigmoid(x) is below 1.1; the gate itself costs a few roundings
    assert np.all(np.abs(out.numpy() - act * u) <= 1.1 * sg * (np.abs(u) + su) + np.abs(act) * su + 1e-6 * np.abs(act * u))
    for b in (da, dw, out):
        b.free()


@pytest.mark.parametrize("fmt,K", [("bf16", 2048), ("bf16", 9216), ("q4", 4096), ("q4", 4736), ("q4", 9216)])
def test_many_steps_to_a_wavefront(lib, orc, fmt, K):
    """Columns that are no multiple of four keep K in one part: a wavefront's steps go through its slots several times (bf16: 8 and
    36 steps in one slot, or four where a block has one row tile; int4: four, five and nine units in two), for one to five (bf16:
    three) row tiles. The sums' order does not depend on the tiles, so the first five rows of every product are the bits of the
    five-row product, which only this kernel forms: the others are formed by it too."""
    N = 33
    A = orc.normal(128 * K, 27).reshape(128, K)
    w, W = _weights(orc, fmt, N, K, 28)
    dw, five = lib.to_device(w), None
    for M in (5, 17, 33, 49, 77, 96, 128):
        print("case gemm_rows long", fmt, M, N, K, flush=True)
        da, out = lib.to_device(A[:M]), lib.to_device(np.full((M, N), np.nan, np.float32))
        (lib.gemm_bf16_nt if fmt == "bf16" else lib.gemm_q4_nt)(da, dw, out, M, N, K)
        got, A64 = out.numpy(), A[:M].astype(np.float64)
        assert np.all(np.abs(got - A64 @ W.T) <= _slack(A64, W, K)), M
        five = got if five is None else five
        assert np.array_equal(got[:5], five), M
        da.free(); out.free()
    dw.free()


@pytest.mark.parametrize("fmt", ["bf16", "q4"])
def test_many_steps_of_wide_gated_tiles(lib, orc, fmt):
    """The same of a gated product wide enough for the widest tiles: 20 steps or five units to a wavefront."""
    ff, K = 4865, 5120
    A = orc.normal(40 * K, 29).reshape(40, K)
    w, W = _weights(orc, fmt, 2 * ff, K, 30)
    p, s = A.astype(np.float64) @ W.T, _slack(A.astype(np.float64), W, K)
    g, u, sg, su = p[:, :ff], p[:, ff:], s[:, :ff], s[:, ff:]
    act = g / (1 + np.exp(-g))
    bound = 1.1 * sg * (np.abs(u) + su) + np.abs(act) * su + 1e-6 * np.abs(act * u)
    dw, five = lib.to_device(w), None
    for M in (5, 20, 40):
        print("case gemm_rows long gated", fmt, M, ff, K, flush=True)
        da, out = lib.to_device(A[:M]), lib.to_device(np.full((M, ff), np.nan, np.float32))
        (lib.gemm_bf16_nt_swiglu if fmt == "bf16" else lib.gemm_q4_nt_swiglu)(da, dw, out, M, ff, K)
        got = out.numpy()
        assert np.all(np.abs(got - (act * u)[:M]) <= bound[:M]), M
        five = got if five is None else five
        assert np.array_equal(got[:5], five), M
        da.free(); out.free()
    dw.free()


# Every block of row tiles and column tiles of the bf16 kernel (1: gated), its wavefronts with more steps than the loop that keeps
# loads in flight needs, some one more than others, in one, two (one row tile, two column tiles) and four slots
TILES = {(0, 1, 1): (3, 17, 2592), (0, 1, 2): (3, 4194, 1568), (0, 1, 3): (3, 8289, 1056), (0, 1, 4): (3, 12664, 3360),
         (0, 2, 1): (33, 17, 1056), (0, 2, 2): (33, 2053, 1056), (0, 2, 3): (17, 8265, 1056), (0, 2, 4): (17, 4120, 3104),
         (0, 3, 1): (65, 17, 1056), (0, 3, 2): (33, 4119, 1056), (0, 3, 3): (65, 4107, 1056), (0, 3, 4): (65, 6165, 1056),
         (0, 4, 1): (150, 17, 1056), (0, 4, 2): (257, 1027, 1056), (0, 4, 3): (49, 8237, 1056), (0, 4, 4): (49, 12386, 1056),
         (0, 5, 1): (200, 1025, 1056), (0, 5, 2): (150, 2726, 1056), (0, 5, 3): (65, 8361, 1056), (0, 5, 4): (65, 4148, 3104),
         (1, 1, 2): (3, 16, 1568), (1, 1, 3): (3, 4134, 1056), (1, 1, 4): (3, 12380, 1056), (1, 2, 2): (33, 17, 1056),
         (1, 2, 3): (17, 4117, 1056), (1, 2, 4): (17, 6223, 1056), (1, 3, 2): (65, 17, 1056), (1, 3, 3): (100, 1367, 1056),
         (1, 3, 4): (65, 3103, 1056), (1, 4, 2): (150, 16, 1056), (1, 4, 3): (49, 4101, 1056), (1, 4, 4): (49, 2088, 3104),
         (1, 5, 2): (150, 1363, 1056), (1, 5, 3): (65, 4137, 1056), (1, 5, 4): (129, 3085, 1056)}


@pytest.mark.parametrize("tile", sorted(TILES))
def test_every_tile(lib, orc, tile):
    """The plan is asked for, so that another estimate cannot move a shape to another tile unseen."""
    gated, TM, TN = tile
    M, N, K = TILES[tile]
    print("case gemm_rows tile", tile, M, N, K, flush=True)
    rows, tm, tn, S, chain = lib.plan_gemm_bf16(M, N, K, bool(gated))
    slots = 4 // TN if TM == 1 and TN <= 2 else 1
    assert (rows, tm, tn) == (1, TM, TN) and chain > 2 * (slots + 1) and -(-K // 32 // S) % 8 != 0
    A = orc.normal(M * K, 37).reshape(M, K)
    w, W = _weights(orc, "bf16", (1 + gated) * N, K, 38)
    p, s = A.astype(np.float64) @ W.T, _slack(A.astype(np.float64), W, K)
    da, dw, out = lib.to_device(A), lib.to_device(w), lib.to_device(np.full((M, N), np.nan, np.float32))
    if gated:
        lib.gemm_bf16_nt_swiglu(da, dw, out, M, N, K)
        g, u, sg, su = p[:, :N], p[:, N:], s[:, :N], s[:, N:]
        act = g / (1 + np.exp(-g))
        assert np.all(np.abs(out.numpy() - act * u) <= 1.1 * sg * (np.abs(u) + su) + np.abs(act) * su + 1e-6 * np.abs(act * u))
    else:
        lib.gemm_bf16_nt(da, dw, out, M, N, K)
        assert np.all(np.abs(out.numpy() - p) <= s)
    for b in (da, dw, out):
        b.free()


@pytest.mark.parametrize("fmt,M,N,K", [("bf16", 40, 130, 896), ("bf16", 150, 130, 896), ("bf16", 300, 1152, 896), ("q4", 40, 130, 896), ("q4", 77, 896, 896), ("q4", 128, 900, 384)])
def test_infinities_and_nan_stay_in_their_rows(lib, orc, fmt, M, N, K):
    """An infinity and a NaN make their rows NaN (an infinity's lower terms are); the other rows keep their bits, also where
    a block multiplies once more for them."""
    print("case gemm_rows not finite", fmt, M, N, K, flush=True)
    A = orc.normal(M * K, 33).reshape(M, K)
    w, _ = _weights(orc, fmt, N, K, 34)
    da, dw, out = lib.to_device(A), lib.to_device(w), lib.empty((M, N))
    call = lib.gemm_bf16_nt if fmt == "bf16" else lib.gemm_q4_nt
    call(da, dw, out, M, N, K)
    clean = out.numpy()
    A[3, 5], A[M - 1, K - 1] = np.inf, np.nan
    call(da.upload(A), dw, out, M, N, K)
    got, rest = out.numpy(), [r for r in range(M) if r not in (3, M - 1)]
    assert np.isnan(got[[3, M - 1]]).all() and np.array_equal(got[rest], clean[rest])
    for b in (da, dw, out):
        b.free()


@pytest.mark.parametrize("fmt,M,N,K", [("bf16", 37, 896, 4864), ("bf16", 77, 896, 4864), ("q4", 20, 896, 4864), ("q4", 77, 896, 4864),
                                         ("bf16", 64, 4608, 3584), ("q4", 128, 4608, 3584),
                                         ("bf16", 200, 896, 4864), ("bf16", 300, 2048, 4096), ("bf16", 130, 5000, 3584)])
def test_recorded_without_scratch(fresh_lib, recorded, orc, fmt, M, N, K):
    """Where the parts of a split K have no room the product is formed in one part, also one that another kernel would have formed
    in parts (the fifth and sixth), and above 128 rows (the last three)."""
    print("case gemm_rows recorded", fmt, M, N, K, flush=True)
    A = orc.normal(M * K, 35).reshape(M, K)
    w, W = _weights(orc, fmt, N, K, 36)
    want, slack = A.astype(np.float64) @ W.T, _slack(A.astype(np.float64), W, K)
    da, dw, out = fresh_lib.to_device(A), fresh_lib.to_device(w), fresh_lib.empty((M, N))
    call = fresh_lib.gemm_bf16_nt if fmt == "bf16" else fresh_lib.gemm_q4_nt
    call(da, dw, out, 1, 16, 128)                  # (the first launch of a library loads its kernels)
    for got in recorded(lambda: call(da, dw, out, M, N, K), out):
        assert np.all(np.abs(got - want) <= slack)
    before = fresh_lib.alloc_calls()
    call(da, dw, out, M, N, K)                     # with scratch to be had: in parts
    assert fresh_lib.alloc_calls() > before and np.all(np.abs(out.numpy() - want) <= slack)
    for b in (da, dw, out):
        b.free()


def test_whole_numbers_are_exact_and_columns_land_where_they_belong(lib, orc):
    """Integer operands give exact integers whatever the order of the sums; every entry of the result differs."""
    rng = np.random.default_rng(31)
    for M, N, K in ((5, 70, 96), (40, 300, 160), (77, 896, 512), (96, 1000, 1024)):
        A = rng.integers(-300, 300, (M, K)).astype(np.float32) + 0.5
        Wf = rng.integers(-60, 60, (N, K)).astype(np.float32)
        da, dw, out = lib.to_device(A), lib.to_device(orc.to_bf16(Wf).reshape(N, K)), lib.empty((M, N))
        lib.gemm_bf16_nt(da, dw, out, M, N, K)
        assert np.array_equal(out.numpy().astype(np.float64), A.astype(np.float64) @ Wf.astype(np.float64).T), (M, N, K)
        for b in (da, dw, out):
            b.free()


@pytest.mark.parametrize("M,N,K", [(65, 896, 896), (77, 301, 896), (96, 260, 2048), (128, 900, 384)])
def test_int4_rows_of_any_magnitude(lib, orc, M, N, K):
    """Above 64 rows an int4 product holds rows of any finite magnitude, denormal ones too, beside ordinary ones and rows
    of zeros, whichever kernel forms it. Results below 2^-126 keep what a denormal holds, once per part of the sum."""
    print("case gemm_rows magnitudes", M, N, K, flush=True)
    w, W = _weights(orc, "q4", N, K, 25)
    da, dw, out, parts = lib.empty((M, K)), lib.to_device(w), lib.empty((M, N)), lib.empty((16, M, N))
    for exps in (np.linspace(-140, 126, M), np.where(np.arange(M) % 9 == 4, 124, 0), np.where(np.arange(M) == M - 1, -130, 0)):
        A = np.clip(orc.normal(M * K, 26).reshape(M, K), -1.9, 1.9).astype(np.float64) * 2.0 ** np.round(exps)[:, None]
        A[3], A[7, : K // 2] = 0.0, 0.0
        A = A.astype(np.float32)
        want, slack = A.astype(np.float64) @ W.T, _slack(A.astype(np.float64), W, K) + 20 * 2.0 ** -149
        lib.gemm_q4_nt(da.upload(A), dw, out, M, N, K)
        assert np.all(np.abs(out.numpy() - want) <= slack)
        n = lib.gemm_q4_nt_parts(da, dw, parts, M, N, K)
        assert np.all(np.abs(parts.numpy()[:n].astype(np.float64).sum(0) - want) <= slack)
    ff = N // 2
    A = np.where(np.abs(exps)[:, None] > 0, A * np.float32(2.0 ** 60), A * np.float32(2.0 ** -120))
    p, s = A.astype(np.float64) @ W[:2 * ff].T, _slack(A.astype(np.float64), W[:2 * ff], K)
    g, u, sg, su = p[:, :ff], p[:, ff:], s[:, :ff], s[:, ff:]
    act, packed = g / (1 + np.exp(-g)), w[:2 * ff * K // 2]
    dw.upload(np.concatenate([packed, w[N * K // 2:][:2 * ff * K // 8]]))
    gated = lib.empty((M, ff))
    lib.gemm_q4_nt_swiglu(da.upload(A), dw, gated, M, ff, K)
    assert np.all(np.abs(gated.numpy() - act * u) <= 1.1 * sg * (np.abs(u) + su) + np.abs(act) * su + 1e-6 * np.abs(act * u) + 2.0 ** -149)
    for b in (da, dw, out, parts, gated):
        b.free()
