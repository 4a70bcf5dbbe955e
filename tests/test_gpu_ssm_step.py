"""GPU parity: the state-space decode step where its blocks take 16 columns of a head and where they take all of it (columns
no multiple of 16, more slices than four per CU), with more and fewer state rows than a block's threads hold, one to
several taps, against the float64 recurrence."""
import numpy as np
import pytest

from test_gpu_state_latent import State, capi, close  # noqa: F401 (capi: a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,N,G,V,taps", [(1, 1, 1, 16, 1), (7, 130, 7, 48, 5), (28, 128, 1, 64, 4), (2, 300, 1, 32, 9), (64, 128, 8, 64, 4), (3, 40, 3, 20, 4),
                                          (520, 8, 4, 32, 3)])
def test_steps(lib, capi, H, N, G, V, taps):
    T = 7
    s = State(lib, capi, H, N, G, V, taps, seed=H)
    u = s.rows(T, N + 1)
    want = s.want(u)
    close(np.stack([s.step(u[t], t) for t in range(T)]), want)
    close(np.stack([s.step(u[T - 1], T - 1) for _ in range(2)]), want[[T - 1, T - 1]])   # a step can be repeated
    p = lib.to_device(np.array([2, 0], np.uint32).view(np.float32))
    for t in range(2):
        s.step(u[t], t)
    close(s.step(u[2], 0, p), want[2])
