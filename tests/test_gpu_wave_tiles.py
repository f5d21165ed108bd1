"""The acoustic step at the edges of its tiles, bit for bit against the oracle.

z extents that leave 0 to 3 cells of the last quad and one quad beyond a
tile, x extents around a tile's rows, y extents of a single plane and of
several uneven chunks, more receivers than one workgroup records, and
wavelets whose field lies in, above and around the denormal range, where the
quotients of the Laplacian round once and no reciprocal may be used carelessly.
"""
import numpy as np
import pytest

import oracle_lib as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz,nx,ny,nb,scale", [
    (56, 8, 3, 4, 1.0),        # one interior tile in z, 16 interior rows
    (57, 9, 2, 4, 1e-36),      # one cell more: a second tile, 17 rows; denormal field
    (58, 24, 1, 4, 1e-30),
    (59, 25, 40, 4, 1e30),
    (24, 41, 61, 5, 1e-38),    # 32-cell z tiles, uneven y chunks
    (25, 33, 90, 4, 1.0),
])
def test_edges_and_ranges(ctx, nz, nx, ny, nb, scale):
    c = orc.acoustic_case(seed=nz, nx=nx, ny=ny, nz=nz, nb=nb, nt=60, spacing=(10.0, 7.3, 12.5))
    c["wavelet"] = (c["wavelet"] * np.float32(scale)).astype(np.float32)
    rng = np.random.default_rng(nz)
    ext = np.array([(n - 1) * d for n, d in zip((nx, ny, nz), c["d"])], np.float32)
    c["rcv"] = (rng.uniform(0, 0.99, (257, 3)).astype(np.float32) * ext).astype(np.float32)
    c["rcv"][0] = c["src"]
    ctx.acoustic_set_model(c["vel"], c["d"], nb=c["nb"], factor=c["factor"], dt=c["dt"])
    seis, uf, _ = ctx.acoustic_shots(c["wavelet"], c["src"][None], c["rcv"], return_ufut=True)
    ref, ref_uf = orc.acoustic_shot(c, want_ufut=True)
    assert np.abs(ref).max() > 0
    assert np.array_equal(seis[0], ref)
    assert np.array_equal(uf, ref_uf)
