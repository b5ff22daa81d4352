"""Iso-values of plus and minus infinity (and NaN, which no sample reaches) over fields with infinite and NaN
samples: the mesh's topology equals the oracle's for rows shorter and longer than a wave, tiles, slabs and the
queue, with the buckets built at once and behind a chain."""
import numpy as np
import pytest

import oracle_api as oa
from test_gpu_parity import gpu, nan_equal

pytestmark = pytest.mark.gpu


def field(shape, seed):
    rng = np.random.default_rng(seed)
    f = rng.uniform(-1, 1, shape).astype(np.float32)
    k = f.size // 3
    f.reshape(-1)[rng.choice(f.size, k, replace=False)] = rng.choice([np.inf, -np.inf], k)
    f.reshape(-1)[rng.choice(f.size, f.size // 30, replace=False)] = np.nan
    return f


@pytest.mark.parametrize("iso", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("shape", [1, 5, 7, 9])
def test_infinite_iso(shape, iso):
    d = gpu()
    d.set_tile_shape(shape)
    try:
        for dims in ((7, 9, 11), (6, 12, 70), (5, 16, 130)):
            f = field(dims, sum(dims))
            for flags in (0, oa.PAD1 | oa.P3X3Y_COLOR | oa.P3333):
                print("infinite iso", shape, iso, dims, flags, flush=True)
                d.extract_raw(f.ctypes.data, dims[::-1], (0, 0, 0), (1, 1, 1), iso, flags)
                m = d.mesh_numpy()
                o = oa.extract(f, (0, 0, 0), (1, 1, 1), iso, flags=flags)
                # (the grid preparation's blend turns an infinite sample into NaN, which reaches no iso-value)
                assert len(o.he) > 0 or iso != -np.inf
                assert np.array_equal(m.halfedges, o.he) and np.array_equal(m.face_attr, o.face_attr)
                assert np.array_equal(m.vertex_flags, o.vflags)
                assert nan_equal("positions", m.positions, o.pos) is None
    finally:
        d.set_tile_shape(0)
