"""Tile edges of the device Podvin & Lecomte solver: its steps visit 8^3 tiles
of the model, so the extents here put one cell less, exactly and one cell more
than whole tiles on each axis, down to the smallest model.  Few shots take eight
waves to a tile, many four; slownesses times spacing below 1e-9 take the general
square roots.  Times must equal the oracle's in every bit.
"""
import numpy as np
import pytest

import oracle_lib as orc

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (7, 8, 9), (8, 8, 8), (9, 16, 17), (15, 24, 7), (25, 9, 23), (3, 33, 4)]


@pytest.mark.parametrize("shots,scale", [(3, 1.0), (300, 1.0), (3, 1e-8), (300, 1e-8)])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("field", ["random", "layers"])
def test_tiles_bit_exact(ctx, shape, shots, scale, field):
    nx, ny, nz = shape
    h = 10.0
    rng = np.random.default_rng(nx * 10000 + ny * 100 + nz + shots)
    if field == "random":
        s = rng.uniform(2e-4, 7e-4, (ny, nx, nz))
    else:       # plane fronts and head waves: equal times, ties between operators
        s = np.broadcast_to(np.where(np.arange(nz) < nz // 2, 6e-4, 2e-4), (ny, nx, nz))
    s = np.ascontiguousarray(s * scale, np.float32)
    ctx.set_model(s, h)
    L = np.array([(nx - 1) * h, (ny - 1) * h, (nz - 1) * h])
    src = rng.uniform(0.0, 1.0, (shots, 3)) * L
    src[0], src[1] = 0.0, L
    src[2] = np.floor(src[2] / h) * h       # on a node: time 0 at the source
    src = np.minimum(src.astype(np.float32), L.astype(np.float32))
    rcv = np.zeros((1, 3), np.float32)
    _, T, _ = ctx.podvin_solve(src, rcv, return_T=True, batch=shots)
    T0 = np.empty((ny, nx, nz), np.float32)
    for i in range(0, shots, 1 if shots < 10 else 97):
        orc.oracle().or_podvin(orc.P(s), nx, ny, nz, h, h, h, float(src[i, 0]), float(src[i, 1]),
                               float(src[i, 2]), orc.P(T0))
        bad = np.argwhere(T[i] != T0)
        assert bad.size == 0, (i, bad[:5])
