"""GPU: a decode step's token travels behind the launches queued before it. Tokens fed with nothing read back in between
give the same bits as tokens after each of which the logits were read (a read waits for the device)."""
import importlib
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("design,name", [("lusadra", "loop_over_everything"), ("girirax", None)])
def test_fed_without_reading(lib, design, name):
    model = importlib.import_module("cpp-tensorlib_amd.model")
    small = importlib.import_module(design + "_models").SMALL
    cfg = small[name or next(iter(small))]
    m = model.Model.random(cfg, seed=3, max_ctx=64, chunk=16)
    t = np.random.default_rng(4).integers(0, m.vocab, 24)
    for _ in range(3):                                   # (the first pass records the step)
        m.reset()
        want = [m.feed([x], [0])[0] for x in t][-1]
        m.reset()
        for x in t[:-1]:
            m.feed([x])
        assert np.array_equal(m.feed(t[-1:], [0])[0], want)
