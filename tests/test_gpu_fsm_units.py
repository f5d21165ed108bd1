"""Accurate_FSM on the device over units of spacing and slowness: 25 m cells,
the coarser ones of crustal models, where 2D roots beside the source have
negative arguments and the method's NaN decides.  Travel times must equal the
oracle's in every bit.
"""
import numpy as np
import pytest

import oracle_lib as orc

pytestmark = pytest.mark.gpu


def _equal_oracle(ctx, shape, d, slow, seed, shots=4):
    nx, ny, nz = shape
    rng = np.random.default_rng(seed)
    s = rng.uniform(*slow, (ny, nx, nz)).astype(np.float32)
    ctx.set_model(s, *d)
    L = (np.array(shape, np.float32) - 1) * np.array(d, np.float32)
    src = np.concatenate([rng.uniform(0, 1, (shots, 3)), [[0, 0, 0], [1, 1, 1], [0.5, 0.5, 0.5]]]) * L
    src = np.minimum(src.astype(np.float32), L)
    _, T, _ = ctx.fsm_solve(src, np.zeros((1, 3), np.float32), return_T=True)
    T0 = np.empty((ny, nx, nz), np.float32)
    for i, p in enumerate(src):
        orc.oracle().or_fsm(orc.P(s), nx, ny, nz, *d, float(p[0]), float(p[1]), float(p[2]),
                            orc.P(T0))
        assert np.array_equal(T[i], T0), (i, T[i].min(), np.abs(T[i] - T0).max())


@pytest.mark.parametrize("v", [1500.0, 3000.0, 6000.0, 12500.0])
@pytest.mark.parametrize("h", [25.0, 50.0, 100.0, 130.0, 200.0, 250.0, 500.0, 1000.0])
def test_spacings_and_speeds(ctx, h, v):
    _equal_oracle(ctx, (21, 19, 17), (h, h, h), (1 / v, 1 / v + 1e-12), int(h + v))
    _equal_oracle(ctx, (21, 19, 17), (h, 0.8 * h, 0.5 * h), (0.9 / v, 1.1 / v), int(h + v))


@pytest.mark.parametrize("d", [(900.0, 1.0, 1.0), (1.0, 1.0, 900.0), (1.0, 30.0, 900.0)])
def test_spacings_far_apart(ctx, d):
    _equal_oracle(ctx, (21, 19, 17), d, (2e-4, 7e-4), 1)
    _equal_oracle(ctx, (5, 7, 90), d, (2e-4, 7e-4), 2)


@pytest.mark.parametrize("d,s", [(9e5, 2e-9),      # root arguments too small for the short form
                                 (9e5, 9.1e-6),    # just large enough
                                 (20.0, 2e-9)])
def test_slownesses_small_against_the_spacing(ctx, d, s):
    _equal_oracle(ctx, (21, 19, 17), (d, 0.9 * d, 0.8 * d), (s, 1.01 * s), 3)


@pytest.mark.parametrize("shape,d,slow", [
    ((13, 15, 6), (911939.0, 3914.5, 443491.0), (4.84, 18.2)),
    ((12, 15, 5), (68431.0, 14860.0, 272024.0), (2.27, 10.7)),
    ((7, 5, 14), (4459.0, 4836.0, 108.6), (721.0, 2209.0)),
    ((11, 9, 8), (10.0, 10.0, 10.0), (500.0, 510.0))])
def test_times_up_to_unreached_ones(ctx, shape, d, slow):
    # times that meet the 1e6 s of unreached cells: sums with those round to
    # multiples of 1/16 s, and some of the method's times come out negative
    _equal_oracle(ctx, shape, d, slow, 4, shots=60)
