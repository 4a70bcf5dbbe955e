"""GPU parity: the bf16 decode product at the edges of its launch rules (rows per CU 16|17, 31|32, 127|128; one to sixteen K
splits, uneven ones too; a last tile and a last chunk that are not full), against float64.

One product is a chain of fewer than K / 64 + 20 fp32 additions per lane and split; the norm forms' x carries a few
roundings of its own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _weight(N, K, seed):
    bits = (np.random.default_rng(seed).standard_normal((N, K)).astype(np.float32) / np.float32(np.sqrt(K))).view(np.uint32) >> 16
    return bits.astype(np.uint16), (bits << 16).astype(np.uint32).view(np.float32)


def _near(got, W, s, slack=0.0):
    W64 = W.astype(np.float64)
    K = W.shape[1]
    assert np.all(np.abs(got - W64 @ s) <= (K / 64 + 40) * 2.0 ** -24 * (np.abs(W64) @ np.abs(s)) + slack)


@pytest.mark.parametrize("N,K", [(3, 8), (1, 4096), (255, 776), (257, 1800), (1025, 6664), (2047, 12288), (2049, 4104), (3073, 768), (3392, 2056),
                                 (4096, 520), (4097, 1536), (7937, 896), (8192, 904), (8193, 2048), (18960, 2056), (32511, 72), (32768, 264)])
def test_plain_and_normed(lib, N, K):
    print("case bf16 rows", N, K, flush=True)
    bits, W = _weight(N, K, N + K)
    g = np.random.default_rng(7)
    x, d, w = (g.standard_normal(K).astype(np.float32) for _ in range(3))
    dx, dd, dw, dW = (lib.to_device(v) for v in (x, d, w, bits))
    y, out = lib.to_device(np.full(N, np.nan, np.float32)), lib.empty(K)
    lib.gemv_bf16_row(dx, dW, y, N, K)
    _near(y.numpy(), W, x.astype(np.float64))
    lib.gemv_bf16_row_rmsnorm(dx, dd, dw, out, dW, y, N, K, 1e-6)
    s = (x + d).astype(np.float64)
    _near(y.numpy(), W, s / np.sqrt(np.mean(s * s) + 1e-6) * w)
    lib.gemv_bf16_row_postnorm(dx, dd, None, dw, K, 1, out, dW, y, N, K, 1e-6)
    n = d.astype(np.float64)
    _near(y.numpy(), W, x + n / np.sqrt(np.mean(n * n) + 1e-6) * w)
    if K % 56 == 0:                                # runs that do not end at 128 values
        r = n.reshape(7, -1)
        lib.gemv_bf16_row_postnorm(dx, dd, None, dw, K, 7, out, dW, y, N, K, 1e-6)
        _near(y.numpy(), W, x + (r / np.sqrt(np.mean(r * r, axis=1, keepdims=True) + 1e-6)).ravel() * w)
    for b in (dx, dd, dw, dW, y, out):
        b.free()


@pytest.mark.parametrize("ff,K", [(1, 64), (1537, 904), (4096, 776), (4097, 2048), (9480, 520), (16200, 136), (130, 8712), (700, 8200)])
def test_gated(lib, ff, K):
    print("case bf16 gated rows", ff, K, flush=True)
    bits, W = _weight(2 * ff, K, ff + K)
    g = np.random.default_rng(8)
    x, d, w = (g.standard_normal(K).astype(np.float32) for _ in range(3))
    gb = g.standard_normal(2 * ff).astype(np.float32)
    dx, dd, dw, dW, dg = (lib.to_device(v) for v in (x, d, w, bits, gb))
    act, out = lib.to_device(np.full(ff, np.nan, np.float32)), lib.empty(K)
    n = d.astype(np.float64)
    s = x + n / np.sqrt(np.mean(n * n) + 1e-6) * w
    lib.gemv_bf16_row_postnorm_geglu(dx, dd, None, dw, out, dW, dg, act, 2 * ff, K, 1e-6)
    W64 = W.astype(np.float64)
    err = (K / 64 + 40) * 2.0 ** -24 * (np.abs(W64) @ np.abs(s) + np.abs(gb))
    z = W64 @ s + gb
    gate = 0.5 * z[:ff] * (1 + np.tanh(np.sqrt(2 / np.pi) * (z[:ff] + 0.044715 * z[:ff] ** 3)))
    # the slope of the gate is below 1.13; the gate itself costs a few roundings
    assert np.all(np.abs(act.numpy() - gate * z[ff:]) <= 1.13 * err[:ff] * (np.abs(z[ff:]) + err[ff:]) + np.abs(gate) * err[ff:] + 1e-6 * (1 + np.abs(gate * z[ff:])))
    t = (x + d).astype(np.float64)
    s = t / np.sqrt(np.mean(t * t) + 1e-6) * w
    lib.gemv_bf16_row_rmsnorm_gateup(dx, dd, dw, out, dW, act, 2 * ff, K, 1e-6)
    z, err = W64 @ s, (K / 64 + 40) * 2.0 ** -24 * (np.abs(W64) @ np.abs(s))
    gate = z[:ff] / (1 + np.exp(-z[:ff]))
    assert np.all(np.abs(act.numpy() - gate * z[ff:]) <= 1.1 * err[:ff] * (np.abs(z[ff:]) + err[ff:]) + np.abs(gate) * err[ff:] + 1e-6 * np.abs(gate * z[ff:]))
    for b in (dx, dd, dw, dW, dg, act, out):
        b.free()


@pytest.mark.parametrize("n,parts,K", [(4096, 8, 4096), (7168, 8, 7168), (256, 2, 264), (384, 3, 520), (1000, 1, 1008), (7, 1, 8), (1200, 8, 1200), (512, 1, 520)])
def test_normed_runs(lib, n, parts, K):
    """Runs of half wavefronts and others, one and several, in rows shorter than the product's K; the row itself is exact to
    the norm's few roundings."""
    print("case bf16 normed runs", n, parts, K, flush=True)
    N = 700
    bits, W = _weight(N, K, n)
    g = np.random.default_rng(9)
    x, d, w, b = (g.standard_normal(K).astype(np.float32) for _ in range(4))
    w[n:] = 0
    for with_x, with_b in ((1, 1), (0, 0)):
        v = (d + with_b * b).astype(np.float64)[:n].reshape(parts, -1)
        s = np.zeros(K)
        s[:n] = (v / np.sqrt(np.mean(v * v, axis=1, keepdims=True) + 1e-6)).ravel() * w[:n]
        s += with_x * x
        dx, dd, db, dw, dW = (lib.to_device(a) for a in (x, d, b, w, bits))
        y, out = lib.to_device(np.full(N, np.nan, np.float32)), lib.to_device(np.full(K, np.nan, np.float32))
        lib.gemv_bf16_row_postnorm(dx if with_x else None, dd, db if with_b else None, dw, n, parts, out, dW, y, N, K, 1e-6)
        # v carries one rounding, its mean square and root (K / 1024 + 20) / 2 together, the product and sum three
        assert np.all(np.abs(out.numpy() - s) <= (K / 2048 + 16) * 2.0 ** -24 * (np.abs(s) + np.abs(with_x * x) + 1))
        _near(y.numpy(), W, s, (K / 2048 + 16) * 2.0 ** -24 * np.abs(W).sum(1).max() * np.abs(s).max())
        for a in (dx, dd, db, dw, dW, y, out):
            a.free()
