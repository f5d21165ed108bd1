"""Travel-time volumes large enough to come back through the pinned slots equal
those of calls small enough not to: with a ragged last chunk, exactly as many
chunks as slots, and the slots reused several times.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,nshot", [((128, 128, 128), 1),      # 8 MiB: the smallest
                                         ((97, 83, 61), 5),         # ragged
                                         ((97, 83, 61), 17)])       # slots reused
def test_volumes_equal_small_calls(ctx, shape, nshot):
    nx, ny, nz = shape
    rng = np.random.default_rng(nshot)
    s = rng.uniform(2e-4, 7e-4, (ny, nx, nz)).astype(np.float32)
    ctx.set_model(s, 10.0, 10.0, 10.0)
    L = (np.array(shape) - 1) * np.float32(10)
    src = (rng.uniform(0, 1, (nshot, 3)) * L).astype(np.float32)
    rcv = (rng.uniform(0, 1, (5, 3)) * L).astype(np.float32)
    picks, T, _ = ctx.fsm_solve(src, rcv, return_T=True)
    assert T.nbytes >= 8 << 20
    _, again, _ = ctx.fsm_solve(src, rcv, return_T=True)
    assert np.array_equal(T, again)
    for i in range(nshot):
        assert np.array_equal(ctx.picks_volume(T[i], (10.0, 10.0, 10.0), rcv), picks[i])
        if nshot > 1:
            _, one, _ = ctx.fsm_solve(src[i:i + 1], rcv, return_T=True)
            assert np.array_equal(T[i], one[0])
