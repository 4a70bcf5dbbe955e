"""GPU: products left as parts, added up by what reads them, for one to sixteen parts and rows at the edges of the blocks'
sizes. The parts are whole numbers, so their sums are exact and the normed rows see the same values as for one part."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [1, 2, 3, 4, 5, 6, 7, 8, 9, 16])
@pytest.mark.parametrize("n", [4, 896, 1024, 1028, 2048, 2052, 4096, 4100])
def test_normed_sums_of_parts(lib, n, S):
    g = np.random.default_rng(n + S)
    rows = 3
    x, w = g.standard_normal((rows, n)).astype(np.float32), g.standard_normal(n).astype(np.float32)
    parts = g.integers(-50, 50, (S, rows, n)).astype(np.float32)
    one = lib.to_device(parts.sum(0))
    dx, dw, dp = lib.to_device(x), lib.to_device(w), lib.to_device(parts)
    out = [[lib.empty((rows, n)) for _ in range(2)] for _ in range(2)]
    for p, k, (xo, h) in ((dp, S, out[0]), (one, 1, out[1])):
        lib.rmsnorm_res_parts(dx, p, k, dw, xo, h, n, 1e-6, rows)
    for a, b in zip(*out):
        assert np.array_equal(a.numpy(), b.numpy())
    s = x.astype(np.float64) + parts.sum(0)
    want = s / np.sqrt(np.mean(s * s, axis=1, keepdims=True) + 1e-6) * w
    # the sum, the mean square of n terms in a tree, root, quotient, two products
    assert np.all(np.abs(out[0][1].numpy() - want) <= (n / 512 + 20) * 2.0 ** -24 * np.abs(want) + 2.0 ** -24 * np.abs(w))
    y = [lib.to_device(x), lib.to_device(x)]
    for p, k, o in ((dp, S, y[0]), (one, 1, y[1])):
        lib.postnorm_res_parts(o, p, k, None, dw, o, n, 1e-6, rows)
    assert np.array_equal(y[0].numpy(), y[1].numpy())
