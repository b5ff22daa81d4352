"""Tile offsets and totals made by the last block of classification (up to 512 tiles) against the scan
that follows it otherwise: tile counts around 1, 256 and 512, tiles without a surface, several
problems, repeated and alternating extractions on one context, against the oracle."""
import numpy as np
import pytest

import oracle_api as oa
from test_gpu_parity import gpu

pytestmark = pytest.mark.gpu

# (nx, ny, nz) by number of 1024-cell tiles: 64 x 16 cells fill one
SIZES = [(65, 17, 2), (65, 17, 3), (65, 17, 4), (65, 17, 256), (65, 17, 257), (65, 17, 258), (65, 17, 512), (65, 17, 513), (65, 17, 514)]


@pytest.mark.parametrize("shape", [1, 2, 3, 4, 5, 6])
def test_around_the_limit(shape):
    d = gpu()
    d.set_tile_shape(shape)
    try:
        for k, (nx, ny, nz) in enumerate(SIZES + SIZES[::-1]):
            rng = np.random.default_rng(k)
            f = np.where(rng.random((nz, ny, nx)) < 0.02, -1.0, 1.0).astype(np.float32)
            f[nz // 3:2 * nz // 3] = 1.0  # whole tiles without a surface
            f[0, 0, 0] = f[-1, -1, -1] = -1.0
            print("totals", shape, nx, ny, nz, flush=True)
            d.extract_raw(f.ctypes.data, (nx, ny, nz), (0, 0, 0), (1, 1, 1), 0.0, 0)
            m = d.mesh_numpy()
            o = oa.extract(f, (0, 0, 0), (1, 1, 1), 0.0, flags=0)
            assert np.array_equal(m.halfedges, o.he) and np.array_equal(m.positions, o.pos), (shape, nx, ny, nz)
    finally:
        d.set_tile_shape(0)
