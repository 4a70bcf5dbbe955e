"""How prompt products are cut into tiles and K splits, asked of the library on the host (for 256 CUs where there is no device):
no plan may trade the error of a sum, which grows with its chain of matrix instructions, for time."""
import random

import pytest


@pytest.fixture(scope="module")
def plans(pkg):
    return pkg.TlHip(init=False)


def _draw(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _ceil(a, b):
    return -(-a // b)


def _filled(M, N, K, gated, parts, cus=256):
    """Slabs of 32 k in a row, summed over the tile columns, where K is split as far as fills the CUs and no further."""
    slabs, cols = K // 32, _ceil(N, 128 if gated else 256)
    tall, low = _ceil(M, 256), _ceil(M, 128)

    def split(n):
        tiles = n * (low if 2 * tall * n <= cus else tall)
        S = min(16, cus // tiles) if N % 4 == 0 and tiles < cus else 1
        while S > 1 and (slabs // S < 8 or (parts and S > parts)):
            S -= 1
        return n * _ceil(slabs, S)

    per_round = cus // tall
    if tall * cols <= cus or per_round == 0 or N % 4 or parts:
        return split(cols)
    whole = cols // per_round * per_round
    return whole * slabs + (split(cols - whole) if whole < cols else 0)


SHAPES = [(512, 4048, 1024, True, 0), (375, 5324, 1248, True, 0), (744, 4824, 1408, False, 16), (615, 3004, 2272, False, 16),
          (996, 4088, 1056, False, 0), (309, 39300, 1056, False, 0), (370, 19908, 10880, True, 0), (300, 18944, 3584, True, 0),
          (122, 4228, 8192, False, 16), (512, 3584, 18944, False, 4), (512, 3584, 3584, False, 1), (65, 130, 64, True, 0),
          (200, 1001, 2048, False, 0), (66000, 4096, 1024, False, 0)]


@pytest.mark.parametrize("M,N,K,gated,parts", SHAPES)
def test_prepared_products_keep_their_chains(plans, M, N, K, gated, parts):
    """Every tile column is in one piece, K is covered, and the chains are no longer than those of the plan that fills the CUs."""
    pieces = plans.plan_gemm_f16w(M, N, K, gated, parts)
    assert 1 <= len(pieces) <= (1 if parts or N % 4 else 2)
    assert sum(p[0] for p in pieces) == _ceil(N, 128 if gated else 256)
    for cols, S, chain, height in pieces:
        assert 1 <= S <= (min(16, parts or 16) if N % 4 == 0 else 1) and height in (128, 256)
        assert (S - 1) * chain < K // 32 <= S * chain
    assert sum(p[0] * p[2] for p in pieces) <= _filled(M, N, K, gated, parts)


def test_prepared_products_keep_their_chains_over_drawn_shapes(plans):
    rng = random.Random(3)
    for _ in range(4000):
        M, N, K = _draw(rng, 65, 1100), _draw(rng, 200, 40000), 32 * _draw(rng, 8, 592)
        if rng.random() < 0.9:
            N = _ceil(N, 4) * 4
        gated, parts = rng.choice([(False, 0), (True, 0), (False, 16), (False, 3)])
        pieces = plans.plan_gemm_f16w(M, N, K, gated, parts)
        assert sum(p[0] * p[2] for p in pieces) <= _filled(M, N, K, gated, parts), (M, N, K, gated, parts)


# M, N, K, gated, room for parts; steps of 32 k in a row and K splits at most
FEW_ROWS = [(24, 1152, 896, False, 16, 1, 4), (100, 1152, 896, False, 16, 1, 4), (24, 896, 896, False, 16, 1, 4), (77, 896, 896, False, 0, 1, 4),
            (40, 896, 4864, False, 16, 2, 16), (77, 896, 4864, False, 16, 2, 16), (16, 4864, 896, True, 0, 4, 1), (77, 4864, 896, True, 0, 4, 1),
            (22, 68, 1600, True, 0, 1, 7), (37, 2048, 8192, False, 16, 4, 16), (127, 248, 1856, True, 0, 1, 8),
            # a block for every CU: no launch to add parts up
            (8, 9000, 2048, False, 0, 8, 1), (32, 9000, 2048, False, 0, 8, 1), (64, 9000, 2048, False, 0, 8, 1), (100, 9000, 2048, False, 0, 8, 1),
            (8, 18960, 2048, False, 0, 8, 1), (32, 18960, 2048, False, 0, 8, 1), (8, 32000, 2048, False, 0, 8, 1), (77, 32000, 2048, False, 0, 8, 1)]


@pytest.mark.parametrize("M,N,K,gated,parts,chain,S", FEW_ROWS)
def test_few_rows_are_split_for_the_error_and_no_further(plans, M, N, K, gated, parts, chain, S):
    got = plans.plan_gemm_bf16(M, N, K, gated, parts)
    assert got[0] == 1 and got[4] <= chain and got[3] <= S, got


def test_few_rows_keep_parts_and_room(plans):
    """A plan's parts are no more than there is room for, and none where N is no multiple of four."""
    rng = random.Random(4)
    for _ in range(4000):
        M, N, K = _draw(rng, 2, 1024), _draw(rng, 16, 40000), 32 * _draw(rng, 4, 592)
        gated, parts = rng.choice([(False, 0), (True, 0), (False, 16), (False, 2), (False, 1)])
        rows, TM, TN, S, chain = plans.plan_gemm_bf16(M, N, K, gated, parts)
        assert 1 <= S <= (1 if N % 4 else min(16, parts or 16)) and chain >= 1, (M, N, K, gated, parts)
        if rows:
            assert 1 <= TM <= 5 and (2 if gated else 1) <= TN <= 4 and chain == _ceil(_ceil(K // 32, S), 8)


# M, N, K, gated, room for parts; us measured in tiles and by the kernel of few rows
MEASURED = [(626, 13780, 640, True, 0, 87.5, 132.2), (270, 18820, 512, False, 16, 26.9, 37.8), (921, 1268, 8128, False, 16, 63.5, 81.9),
            (366, 4728, 3456, False, 16, 43.5, 57.3), (242, 4608, 3584, False, 16, 33.1, 44.6), (476, 2048, 4096, False, 16, 34.0, 43.7),
            (108, 21844, 1344, False, 16, 31.7, 41.9), (512, 896, 6656, False, 16, 29.3, 34.3),
            (300, 1152, 896, False, 16, 21.3, 7.2), (202, 5886, 384, False, 16, 24.2, 11.5), (150, 896, 4864, False, 16, 22.3, 10.5),
            (256, 4864, 896, True, 0, 28.4, 24.8), (77, 4864, 896, True, 0, 24.9, 10.6), (64, 18944, 3584, True, 0, 106.9, 88.7),
            (77, 32000, 2048, False, 0, 56.1, 46.6), (32, 9000, 2048, False, 0, 18.8, 14.8)]


@pytest.mark.parametrize("M,N,K,gated,parts,tiles,rows", MEASURED)
def test_the_faster_kernel_is_chosen(plans, M, N, K, gated, parts, tiles, rows):
    assert plans.plan_gemm_bf16(M, N, K, gated, parts)[0] == (rows < tiles)


# M, N, K, gated, room for parts; row and column tiles of a block, us measured with them and with the tiles that an estimate took which
# had other numbers of blocks on a CU than the kernel's LDS allows
TILES = [(86, 5216, 416, True, 0, 2, 4, 6.75, 8.21), (24, 13272, 320, True, 0, 2, 4, 6.58, 8.00), (178, 2976, 256, False, 0, 3, 3, 4.28, 5.10),
         (142, 18080, 352, True, 0, 3, 3, 22.9, 27.9), (186, 8988, 352, False, 0, 3, 3, 9.30, 11.4), (18, 38236, 384, True, 0, 2, 4, 16.2, 20.4)]


@pytest.mark.parametrize("M,N,K,gated,parts,TM,TN,us,other", TILES)
def test_blocks_on_a_cu_are_those_its_lds_takes(plans, M, N, K, gated, parts, TM, TN, us, other):
    assert us < other and plans.plan_gemm_bf16(M, N, K, gated, parts)[:3] == (1, TM, TN)


@pytest.mark.parametrize("M,N,K", [(129, 999, 8192), (200, 1151, 4864), (150, 3585, 3584), (1000, 301, 12288)])
def test_a_k_that_cannot_be_split_has_no_longer_chains_above_128_rows(plans, M, N, K):
    """The tiles cannot split it either: theirs would be all of K (129 x 999 x 8192 369 us, 26 here)."""
    rows, _, _, S, chain = plans.plan_gemm_bf16(M, N, K)
    assert (rows, S) == (1, 1) and chain == _ceil(K // 32, 8)


@pytest.mark.parametrize("M,N,K", [(1 << 31, 1 << 31, 128), (1 << 30, 64, 128), (64, 1 << 30, 128), (1 << 29, 1 << 29, 128), (64, 64, 1 << 40)])
def test_plans_refuse_what_no_product_takes(plans, M, N, K):
    """With an error: the bytes of the first wrap to none, by which the room for parts was divided."""
    for ask in (plans.plan_gemm_bf16, plans.plan_gemm_f16w):
        for parts in (0, 16):
            with pytest.raises(Exception, match="dimension too large"):
                ask(M, N, K, False, parts)
