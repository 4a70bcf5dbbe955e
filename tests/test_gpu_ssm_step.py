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


@pytest.mark.parametrize("H,N,G,V,taps", [(4, 200, 2, 32, 4), (2, 300, 1, 16, 4), (2, 512, 2, 16, 4), (2, 260, 1, 32, 6), (512, 8, 1, 16, 4), (256, 8, 256, 32, 4),
                                          (3, 20, 1, 16, 64)])
def test_sliced_steps_at_their_limits(lib, capi, H, N, G, V, taps):
    """Slices of 16 columns: two state rows to a thread and more, more channels than threads with four taps and with others, as many
    blocks as are taken, all heads in one group and each in its own, the most taps; chunks and steps over one state."""
    print("case ssm limits", H, N, G, V, taps, flush=True)
    test_steps(lib, capi, H, N, G, V, taps)
    T = 23 if taps < 64 else 140
    s = State(lib, capi, H, N, G, V, taps, seed=H + 1)
    u = s.rows(T, N + 2)
    got, t = [], 0
    for n in (1, 1, 1, 5, 1, 2, 1, 1, T - 17, 1, 1, 1, 1):
        got.append(s.chunk(u[t:t + n], t) if n > 1 else s.step(u[t], t)[None])
        t += n
    assert t == T
    close(np.concatenate(got), s.want(u))
