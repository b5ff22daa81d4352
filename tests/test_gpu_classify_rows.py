"""Classification takes the x + 1 corners of a wave's 64 consecutive cells from its neighbours' ballots
where rows have 64 cells or more, and reads eight corners per cell where they are shorter: rows
around one and two waves, row ends in every lane, a last tile that ends inside a wave, NaN samples, for
every tile shape, against the oracle."""
import numpy as np
import pytest

import oracle_api as oa
from test_gpu_parity import gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [1, 2, 3, 4, 5, 6, 9])
def test_rows(shape):
    d = gpu()
    rng = np.random.default_rng(shape)
    d.set_tile_shape(shape)
    try:
        for nx in (3, 64, 65, 66, 67, 128, 129, 130, 131, 257, 300):
            for ny, nz in ((2, 2), (3, 5), (9, 4)):
                f = rng.uniform(-1, 1, (nz, ny, nx)).astype(np.float32)
                if nx == 131:
                    f.reshape(-1)[rng.choice(f.size, 9, replace=False)] = np.nan
                    f.reshape(-1)[rng.choice(f.size, 9, replace=False)] = 0.0
                print("rows", shape, nx, ny, nz, flush=True)
                d.extract_raw(f.ctypes.data, (nx, ny, nz), (0, 0, 0), (1, 1, 1), 0.0, 0)
                m = d.mesh_numpy()
                o = oa.extract(f, (0, 0, 0), (1, 1, 1), 0.0, flags=0)
                assert np.array_equal(m.halfedges, o.he) and np.array_equal(m.face_attr, o.face_attr), (shape, nx, ny, nz)
                assert np.array_equal(m.positions.view(np.uint32)[~np.isnan(o.pos)], o.pos.view(np.uint32)[~np.isnan(o.pos)])
    finally:
        d.set_tile_shape(0)
