"""Arrival ordering at the shot counts where the number of words holding a
shot's smallest key changes (eight up to 32 shots, four, two, one from 129 on),
for both block edges, both visit forms and the caller-predicted start.  With eps
= 0 every visit order ends at the fixed point of the update, so the ordered
solves equal the unordered one but for the rounding of the last updates: at most
a few units in the last place of times below 0.5 s per cell crossed, 1e-6 s.
"""
import numpy as np
import pytest

from seismic_tomography_3d_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block,sweep", [(8, 0), (8, 1), (4, 0)])
@pytest.mark.parametrize("shots", [1, 32, 33, 64, 65, 128, 129, 260])
def test_ordered_equals_unordered(ctx, shots, block, sweep):
    nx, ny, nz, h = 27, 33, 18, 12.5
    vel = synth.layered_model(nx, ny, nz, h, n_layers=3, n_anom=2, seed=4)
    ctx.set_model(1.0 / vel, h)
    src = synth.random_sources(shots, nx, ny, h, 0.0, (nz - 1) * h, seed=shots)
    kw = dict(block=block, sweep=sweep, eps=0.0, batch=shots)
    _, T0, _ = ctx.fim_solve(src, None, return_T=True, **kw)
    assert T0.max() < 0.5
    for band in (0.0, 0.01):
        _, T1, st = ctx.fim_solve(src, None, return_T=True, order=1, band=band, **kw)
        assert np.abs(T1 - T0).max() <= 1e-6
        if band:
            assert st["deferred"] > 0
    _, T2, _ = ctx.fim_solve_warm(src, None, T0, return_T=True, warm_values=0, **kw)
    assert np.abs(T2 - T0).max() <= 1e-6
    _, T3, _ = ctx.fim_solve_warm(src, None, T0, return_T=True, warm_values=0, order=2, **kw)
    assert np.abs(T3 - T0).max() <= 1e-6
