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
