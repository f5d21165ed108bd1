"""Block edges of the device Accurate_FSM: sweeps run in blocks of 8 x 8
columns by up to 14 cells of z counted from each shot's own start corner, so
the padded extents here put one cell less, exactly, and one cell more than a
block on each axis, down to the smallest model.  Travel times must equal the
oracle's in every bit, in the ordinary range of units (short square roots and
quotients, operators that cannot win left out) and outside it (slownesses or
spacing ratios that take the update as the method's code has it).
"""
import numpy as np
import pytest

import oracle_lib as orc

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (6, 7, 12), (7, 6, 13), (8, 9, 14), (15, 14, 27), (16, 22, 28), (23, 15, 29),
          (3, 40, 5)]
UNITS = [((25.0, 25.0, 25.0), 1.0),      # short forms
         ((10.0, 25.0, 4.0), 1.0),
         ((25.0, 25.0, 25.0), 1e-7),     # slownesses below 1e-9 s/m: general form
         ((2000.0, 1.5, 1.0), 1.0)]      # spacings further apart than 1000: general form


@pytest.mark.parametrize("units", UNITS)
@pytest.mark.parametrize("shape", SHAPES)
def test_blocks_bit_exact(ctx, shape, units):
    nx, ny, nz = shape
    (dx, dy, dz), scale = units
    rng = np.random.default_rng(nx * 10000 + ny * 100 + nz)
    s = (rng.uniform(2e-4, 7e-4, (ny, nx, nz)) * scale).astype(np.float32)
    ctx.set_model(s, dx, dy, dz)
    L = np.array([(nx - 1) * dx, (ny - 1) * dy, (nz - 1) * dz])
    src = np.concatenate([rng.uniform(0.0, 1.0, (3, 3)), [[0, 0, 0], [1, 1, 1], [1, 0, 0.5]]]) * L
    src = np.minimum(src.astype(np.float32), L.astype(np.float32))
    rcv = np.zeros((1, 3), np.float32)
    _, T, _ = ctx.fsm_solve(src, rcv, return_T=True)
    T0 = np.empty((ny, nx, nz), np.float32)
    for i, p in enumerate(src):
        orc.oracle().or_fsm(orc.P(s), nx, ny, nz, dx, dy, dz, float(p[0]), float(p[1]),
                            float(p[2]), orc.P(T0))
        assert np.array_equal(T[i], T0), (i, np.abs(T[i] - T0).max())
