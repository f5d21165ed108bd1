"""Full sweeps of the device Accurate_FSM walk only the blocks a test of all
cells has marked and those behind a changed face.  Models whose fronts wind
through the blocks -- a fast channel folded through slow rock, random
contrasts of 20 to 1 -- keep changing blocks that the test could not mark, for
shot counts around the eight lists of a diagonal, alone and in batches that
reuse the lists.  Travel times must equal the oracle's in every bit.
"""
import numpy as np
import pytest

import oracle_lib as orc

pytestmark = pytest.mark.gpu


def _channel(nx, ny, nz):
    s = np.full((ny, nx, nz), 2e-3, np.float32)
    for y in range(1, ny, 4):                    # galleries along x ...
        s[y, 1:-1, 2] = 1e-4
        side = nx - 2 if (y // 4) % 2 == 0 else 1
        s[y:y + 4, side, 2] = 1e-4               # ... joined at alternating ends
    s[ny // 2, nx // 2, 2:] = 1e-4
    return s


def _contrast(nx, ny, nz):
    rng = np.random.default_rng(nx + ny + nz)
    return np.where(rng.random((ny, nx, nz)) < 0.5, 1e-4, 2e-3).astype(np.float32)


@pytest.mark.parametrize("nshot,batch", [(1, 0), (7, 0), (8, 0), (9, 4), (17, 0)])
@pytest.mark.parametrize("model", [_channel, _contrast])
@pytest.mark.parametrize("shape,d", [((40, 33, 30), (25.0, 25.0, 25.0)),
                                     ((17, 41, 16), (2000.0, 1.5, 1.0))])   # general form
def test_winding_fronts(ctx, shape, d, model, nshot, batch):
    nx, ny, nz = shape
    s = model(nx, ny, nz)
    ctx.set_model(s, *d)
    L = ((np.array(shape) - 1) * np.array(d)).astype(np.float32)
    rng = np.random.default_rng(nshot)
    src = (rng.uniform(0, 1, (nshot, 3)) * L).astype(np.float32)
    src[0] = 0
    _, T, _ = ctx.fsm_solve(src, np.zeros((1, 3), np.float32), return_T=True, batch=batch)
    T0 = np.empty((ny, nx, nz), np.float32)
    for i, p in enumerate(src):
        orc.oracle().or_fsm(orc.P(s), nx, ny, nz, *d, float(p[0]), float(p[1]), float(p[2]),
                            orc.P(T0))
        assert np.array_equal(T[i], T0), (i, np.abs(T[i] - T0).max())
