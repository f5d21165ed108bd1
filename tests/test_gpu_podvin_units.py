"""Podvin & Lecomte on the device over units of spacing and slowness, from
products of both far below a second to times beyond the 1e6 s that stand for
"not reached" (the front stops there; a source further than that from its node
reaches nothing).  Times must equal the oracle's in every bit.
"""
import numpy as np
import pytest

import oracle_lib as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,scale", [(10.0, 1e-12), (25.0, 1e-4), (1000.0, 1.0), (10.0, 1e6),
                                     (10.0, 2e7), (10.0, 2e8), (10.0, 1e9), (10.0, 1e12)])
def test_units_bit_exact(ctx, h, scale):
    nx, ny, nz = 19, 13, 11
    rng = np.random.default_rng(5)
    s = (rng.uniform(2e-4, 7e-4, (ny, nx, nz)) * scale).astype(np.float32)
    ctx.set_model(s, h)
    L = ((np.array([nx, ny, nz]) - 1) * h).astype(np.float32)
    src = (rng.uniform(0.0, 1.0, (24, 3)) * L).astype(np.float32)
    src[0] = 0.0
    src[1] = np.floor(src[1] / h) * h
    src = np.minimum(src, L)
    _, T, _ = ctx.podvin_solve(src, np.zeros((1, 3), np.float32), return_T=True, batch=24)
    T0 = np.empty((ny, nx, nz), np.float32)
    for i, p in enumerate(src):
        orc.oracle().or_podvin(orc.P(s), nx, ny, nz, h, h, h, float(p[0]), float(p[1]),
                               float(p[2]), orc.P(T0))
        bad = np.argwhere(T[i] != T0)
        assert bad.size == 0, (i, bad[:5], T[i].max(), T0.max())
