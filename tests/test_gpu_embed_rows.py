"""GPU: embedding rows by ids that ride with the launch (tlhip_embed_rows): widening is exact, so the rows are equal bit for
bit; widths of whole and broken 16 bytes, more ids than one launch takes, ids outside the table refused."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("T,hidden,vocab", [(1, 896, 512), (8, 3584, 40), (9, 896, 40), (3, 900, 77), (768, 8, 300), (769, 2056, 5), (2000, 33, 1000)])
def test_rows(lib, f16, T, hidden, vocab):
    g = np.random.default_rng(T)
    bits = g.integers(0, 1 << 16, (vocab, hidden), dtype=np.uint16)
    bits[(bits & 0x7c00) == 0x7c00] &= 0x83ff if f16 else 0xffff        # (f16 infinities and NaN: compared by value below only for bf16)
    ids = g.integers(0, vocab, T)
    ids[0], ids[-1] = vocab - 1, 0
    want = bits.view(np.float16).astype(np.float32).view(np.uint32) if f16 else bits.astype(np.uint32) << 16
    table, out = lib.to_device(bits), lib.to_device(np.full((T, hidden), np.nan, np.float32))
    lib.embed_rows(table, lib.T_F16 if f16 else lib.T_BF16, ids, out, hidden, vocab)
    assert np.array_equal(out.numpy().view(np.uint32), want[ids])
    table.free(); out.free()


def test_refused(lib, pkg):
    table, out = lib.empty(64 * 8, np.uint16), lib.to_device(np.full((2, 8), 7.0, np.float32))
    for ids, kind in (([0, 64], lib.T_BF16), ([-1, 0], lib.T_F16), ([0, 1 << 40], lib.T_F16), ([0, 1], lib.T_F32), ([], lib.T_F16)):
        with pytest.raises(pkg.TlHipError):
            lib.embed_rows(table, kind, ids, out, 8, 64)
    assert np.all(out.numpy() == 7.0)
    table.free(); out.free()
