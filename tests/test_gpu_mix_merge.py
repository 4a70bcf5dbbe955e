"""GPU: the output product of a layer that merges the splits of its windowed attention while it stages its input
(tlhip_mix_step_open, tlhip_gemv_bf16_row_mix): the same arithmetic as the merge launch and the plain product, so the same
bits; splits that hold no key yet, columns ahead of and behind the attention's, rows longer than a block holds up front."""
import ctypes as C
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    return importlib.import_module("cpp-tensorlib_amd.capi")


def rng(seed):
    return np.random.default_rng(seed)


def setting(lib, capi, H, G, dim, window, gate, first, tail):
    ld = lib.c.tlhip_window_ring_ld(dim)
    ring = lib.to_device(rng(7).standard_normal((G, (window + 31) // 32 * 32, ld)).astype(np.float32))
    q, k = H * dim, G * dim
    at = capi.WindowAttn(heads=H, kv_heads=G, dim=dim, window=window, q_off=0, k_off=q, gate_off=q + k if gate else -1, y_off=first,
                         ring=ring.ptr, ring_rows=(window + 31) // 32 * 32, ring_ld=ld, scale=dim ** -0.5, temp_coef=0.3, temp_every=16,
                         slope_exp=8.0, out_scale=0.7)
    return at, ring, 2 * q + k, (first + q + tail + 7) // 8 * 8


@pytest.mark.parametrize("H,G,dim,window,gate,first,tail,n", [
    (16, 4, 128, 1024, True, 0, 10240, 2048),     # 8 splits, one tile of rows a block
    (16, 4, 128, 1024, False, 8, 512, 300),       # columns ahead; no gate
    (28, 4, 128, 1024, True, 0, 16896, 3584),     # as many columns as it takes
    (6, 2, 128, 400, True, 4, 4, 40),             # 4 splits, short blocks: columns past what a thread asks for up front
    (40, 4, 64, 2048, True, 1004, 100, 5000),     # more columns than threads, K split
    (5, 5, 36, 1100, True, 0, 0, 17),             # heads of a width that no vector divides
    (6, 3, 4, 2048, True, 4, 4, 40),              # heads of a single float4, and of two
    (70, 7, 4, 1600, False, 0, 16, 300),
    (6, 2, 8, 4096, True, 0, 0, 33),
])
def test_same_bits(lib, capi, H, G, dim, window, gate, first, tail, n):
    at, ring, width, K = setting(lib, capi, H, G, dim, window, gate, first, tail)
    assert lib.c.tlhip_mix_open(C.byref(at), K)
    nb = lib.mix_partials_bytes(at)
    W = lib.to_device((rng(3).standard_normal((n, K)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16))
    y0 = rng(5).standard_normal(K).astype(np.float32)
    for pos in (0, 3, 130, window // 2, window - 1, 3 * window + 5):
        if at.ring_rows < min(window, pos + 1):
            continue
        u = lib.to_device(rng(pos).standard_normal((width + 3) // 4 * 4).astype(np.float32))
        outs = []
        for opened in (False, True):
            parts, y, out = lib.empty(nb // 4), lib.to_device(y0), lib.empty(n)
            if opened:
                y0_attn = y0.copy()
                y0_attn[first:first + H * dim] = np.nan          # not read
                y.upload(y0_attn)
                assert lib.c.tlhip_mix_step_open(u.ptr, y.ptr, C.byref(at), None, None, pos, None, parts.ptr, nb) == 0
                assert lib.c.tlhip_gemv_bf16_row_mix(y.ptr, u.ptr, C.byref(at), parts.ptr, nb, W.ptr, out.ptr, n, K) == 0
            else:
                lib.mix_step(u, y, at, None, None, pos, None, parts)
                lib._chk(lib.c.tlhip_gemv_bf16_row(y.ptr, W.ptr, out.ptr, n, K))
            outs.append(out.numpy().view(np.uint32).copy())
            for b in (parts, y, out):
                b.free()
        assert np.all(np.isfinite(outs[0].view(np.float32))) and np.array_equal(outs[0], outs[1]), (pos, np.sum(outs[0] != outs[1]))
        u.free()
    W.free(); ring.free()


def test_refused(lib, capi):
    W, out = lib.empty(64 * 4096, np.uint16), lib.empty(64)
    u, y = lib.empty(16384), lib.empty(4096)

    def rc(at, K=4096, parts=None, nb=None):
        need = lib.mix_partials_bytes(at)
        p = parts or lib.empty(max(need // 4, 4))
        return lib.c.tlhip_gemv_bf16_row_mix(y.ptr, u.ptr, C.byref(at), p.ptr, need if nb is None else nb, W.ptr, out.ptr, 64, K)
    at, ring, _, _ = setting(lib, capi, 16, 4, 128, 1024, True, 0, 0)
    assert rc(at, nb=lib.mix_partials_bytes(at) - 4) != 0                   # partials too small
    assert rc(at, K=2040) != 0                                              # columns past K
    for name, value in (("y_off", 2), ("gate_off", 2562), ("window", 4096), ("window", 100)):
        keep = getattr(at, name)
        setattr(at, name, value)
        assert not lib.c.tlhip_mix_open(C.byref(at), 4096) and rc(at) != 0        # its own merge launch, or none at all
        setattr(at, name, keep)
    assert lib.c.tlhip_mix_open(C.byref(at), 20480) and not lib.c.tlhip_mix_open(C.byref(at), 20488) and not lib.c.tlhip_mix_open(None, 4096)
