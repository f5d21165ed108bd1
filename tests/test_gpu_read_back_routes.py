"""Every way a large travel-time volume takes to the caller: through the pinned
slots from each solver and from the forward pass, and directly where the
destination is pinned or device memory.  The same volumes must come back: from
calls of single shots, too small for the slots, from the direct route, and as
the picks of the same call, taken from the volumes on the device, have them.
"""
import ctypes

import numpy as np
import pytest

from seismic_tomography_3d_amd import _lib

pytestmark = pytest.mark.gpu

H = 10.0
SHAPE, SHOTS = (97, 83, 61), 6      # 11.8 MB: eleven chunks and part of one


def _setup(ctx, shape, shots, nrcv, seed=3):
    nx, ny, nz = shape
    rng = np.random.default_rng(seed)
    ctx.set_model(rng.uniform(2e-4, 7e-4, (ny, nx, nz)).astype(np.float32), H)
    L = (np.array(shape) - 1) * np.float32(H)
    return ((rng.uniform(0, 1, (shots, 3)) * L).astype(np.float32),
            (rng.uniform(0, 1, (nrcv, 3)) * L).astype(np.float32))


@pytest.mark.parametrize("solver", ["fsm_solve", "podvin_solve"])
def test_solvers_equal_single_shots(ctx, solver):
    src, rcv = _setup(ctx, SHAPE, SHOTS, 5)
    solve = getattr(ctx, solver)
    _, T, _ = solve(src, rcv, return_T=True)
    assert T.nbytes >= 8 << 20
    for i in range(SHOTS):
        _, one, _ = solve(src[i:i + 1], rcv, return_T=True)
        assert np.array_equal(T[i], one[0])


@pytest.mark.parametrize("order", [0, 1])
def test_fim_equals_its_picks(ctx, order):
    src, rcv = _setup(ctx, SHAPE, SHOTS, 20000)
    picks, T, _ = ctx.fim_solve(src, rcv, return_T=True, order=order)
    assert T.nbytes >= 8 << 20
    for i in range(SHOTS):
        assert np.array_equal(ctx.picks_volume(T[i], (H, H, H), rcv), picks[i])


@pytest.mark.parametrize("eikonal", [0, 1, 2])
def test_forward_equals_its_picks(ctx, eikonal):
    src, rcv = _setup(ctx, SHAPE, SHOTS, 300)
    ctx.tomo_set_grid(5 * H)
    ctx.tomo_set_eikonal(eikonal)
    try:
        dcal, _, _, T = ctx.forward(src, rcv, return_T=True)
    finally:
        ctx.tomo_set_eikonal(1)
    for i in range(SHOTS):
        assert np.array_equal(ctx.picks_volume(T[i], (H, H, H), rcv), dcal[i])
    if eikonal != 1:
        solve = ctx.fsm_solve if eikonal == 2 else ctx.podvin_solve
        for i in range(SHOTS):
            assert np.array_equal(T[i], solve(src[i:i + 1], rcv, return_T=True)[1][0])


def _runtime():
    """The HIP runtime the library is linked to."""
    with open("/proc/self/maps") as f:
        for line in f:
            if "libamdhip64" in line:
                return ctypes.CDLL(line.split()[-1])
    raise RuntimeError("no HIP runtime loaded")


@pytest.mark.parametrize("shape,shots", [((128, 128, 128), 1),     # as many chunks as slots
                                         (SHAPE, SHOTS)])
@pytest.mark.parametrize("where", ["pinned", "device"])
def test_direct_destinations(ctx, where, shape, shots):
    src, rcv = _setup(ctx, shape, shots, 5)
    picks, T, _ = ctx.fsm_solve(src, rcv, return_T=True)
    lib, hip = _lib.load(), _runtime()
    p, n = ctypes.c_void_p(), ctypes.c_size_t(T.nbytes)
    if where == "pinned":
        assert hip.hipHostMalloc(ctypes.byref(p), n, 0) == 0
    else:
        assert hip.hipMalloc(ctypes.byref(p), n) == 0
    got = np.empty_like(picks)
    fp = ctypes.POINTER(ctypes.c_float)
    rc = lib.st_fsm_solve(ctx.h, src.ctypes.data_as(fp), shots, rcv.ctypes.data_as(fp), len(rcv),
                          got.ctypes.data_as(fp), ctypes.cast(p, fp), 0, None)
    back = np.empty_like(T)
    if rc == 0:
        assert hip.hipMemcpy(ctypes.c_void_p(back.ctypes.data), p, n, 4) == 0
    assert (hip.hipHostFree if where == "pinned" else hip.hipFree)(p) == 0
    assert rc == 0
    assert np.array_equal(got, picks)
    assert np.array_equal(back, T)
