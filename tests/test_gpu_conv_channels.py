"""Weight gradient of a convolution whose output channels do not fill the tiles
of 16 that the kernel takes: 20 (the reads of four channels at a time end inside
a tile), 18 (reads by single channels) and 4, on a cube of part bricks.  The
library's own function, on buffers without room behind the last voxel, against
torch in 64 bits from the same BF16 values.  Tolerance: FP32 sums of at most
2 x 9^3 products, 2 x 9^3 x 2^-24 = 9e-5 of the sum of their magnitudes.
"""
import ctypes

import numpy as np
import pytest
import torch

from seismic_tomography_3d_amd import _lib

pytestmark = pytest.mark.gpu

FUNC = "_ZN2st2nn20conv_backward_weightEP12ihipStream_tPKfPKtPfiiiii"


def _runtime():
    """The HIP runtime the library is linked to."""
    with open("/proc/self/maps") as f:
        for line in f:
            if "libamdhip64" in line:
                return ctypes.CDLL(line.split()[-1])
    raise RuntimeError("no HIP runtime loaded")


@pytest.mark.parametrize("cout", [20, 18, 4])
@pytest.mark.parametrize("cin", [16, 6])
def test_weight_gradient(ctx, cin, cout):
    lib = _lib.load()
    hip = _runtime()
    ns, e, ks = 2, 9, 3
    rng = np.random.default_rng(cin + cout)
    X = torch.tensor(rng.normal(0, 1, (ns, e, e, e, cin)), dtype=torch.float32)
    D = torch.tensor(rng.normal(0, 1, (ns, e, e, e, cout))).to(torch.bfloat16)
    X = X.to(torch.bfloat16).to(torch.float32)
    dW = np.zeros((ks ** 3, cin, cout), np.float32)
    host = [np.ascontiguousarray(X.numpy()), np.ascontiguousarray(D.view(torch.int16).numpy()), dW]
    dev = []
    for a in host:
        p = ctypes.c_void_p()
        assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(a.nbytes)) == 0
        assert hip.hipMemcpy(p, ctypes.c_void_p(a.ctypes.data), ctypes.c_size_t(a.nbytes), 1) == 0
        dev.append(p)
    f = getattr(lib, FUNC)
    f.restype = None
    f(None, *dev, ns, e, cin, cout, ks)
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemcpy(ctypes.c_void_p(dW.ctypes.data), dev[2], ctypes.c_size_t(dW.nbytes), 2) == 0
    for p in dev:
        assert hip.hipFree(p) == 0

    def grad(x, d):
        g = torch.nn.grad.conv3d_weight(x.double().permute(0, 4, 1, 2, 3),
                                        (cout, cin, ks, ks, ks),
                                        d.double().permute(0, 4, 1, 2, 3), padding=1)
        return g.permute(2, 3, 4, 1, 0).reshape(ks ** 3, cin, cout).numpy()
    g0, mag = grad(X, D), grad(X.abs(), D.abs())
    assert (np.abs(dW - g0) <= 9e-5 * mag).all()
