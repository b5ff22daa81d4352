"""The adjoint's per-point pass at its edges: single layers (every padded copy of a point),
grids of one cell, partial blocks, dense surfaces; with and without padding and refinement,
overwriting and accumulating.  Reference and tolerance as in test_gpu_adjoint.py (FP64
scatter over every vertex, 1e-4 of the gradient's norm); points with no vertex around keep
exactly 0, or exactly their value."""
import numpy as np
import pytest

import oracle_api as oa
from test_gpu_adjoint import enumerate_vertices, input_gradient64, processed_gradient64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("dims,pad,refinement", [((1, 1, 7), True, 0), ((5, 1, 4), True, 0), ((2, 2, 2), False, 0), ((2, 2, 2), True, 0),
                                                 ((3, 9, 1), True, 1), ((17, 6, 5), False, 0), ((33, 7, 6), True, 0), ((6, 5, 7), False, 2),
                                                 ((16, 16, 17), True, 0)])
def test_points_match_fp64(dims, pad, refinement, accumulate):
    import torch

    import manifolddmc_amd as mdmc
    nx, ny, nz = dims
    rng = np.random.default_rng(nx + 10 * ny + 100 * nz)
    field = rng.uniform(-1, 1, (nz, ny, nx)).astype(np.float32)
    if nz > 8:  # half of the grid without surface
        field[nz // 2:] = np.abs(field[nz // 2:]) + 0.1
    origin, delta = (0.1, -0.2, 0.3), (0.5, 0.25, 0.75)
    d = mdmc.DualMarchingCubes()
    try:
        t = torch.from_numpy(field).cuda()
        torch.cuda.synchronize()
        print("adjoint points", dims, pad, refinement, accumulate, flush=True)
        d.extract_raw(t.data_ptr(), dims, origin, delta, 0.0, mdmc.RECORD_ADJOINT | (mdmc.PAD1 if pad else 0), refinement, True)
        V = d.info()[0]
        gpos = rng.normal(size=(V, 3)).astype(np.float32)
        start = rng.normal(size=field.shape).astype(np.float32)
        gd, out = torch.from_numpy(gpos).cuda(), torch.from_numpy(start).cuda()
        torch.cuda.synchronize()
        d.backward(gd.data_ptr() if V else 0, out.data_ptr(), accumulate)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
    finally:
        d.close()
    o = oa.extract(field, origin, delta, 0.0, flags=oa.PAD1 if pad else 0, refinement=refinement, want_grid=True)
    verts = enumerate_vertices(o.grid, 0.0)
    assert len(verts) == V
    dproc = processed_gradient64(o.grid.astype(np.float64), verts, 0.0, np.asarray(o.grid_delta, np.float64), gpos.astype(np.float64))
    ref = input_gradient64(dproc, field.shape, refinement, 1 if pad else 0)
    base = start.astype(np.float64) if accumulate else 0.0
    assert np.linalg.norm(got - (base + ref)) <= 1e-4 * max(np.linalg.norm(ref), 1e-30) + (1e-6 * np.linalg.norm(base) if accumulate else 0.0)
    still = ref == 0
    assert np.array_equal(got[still], start[still] if accumulate else np.zeros(still.sum(), np.float32))
