"""Padding of fields with and without values that need the exact blend (-0, infinities, huge
values), call after call on one context: the exact pass runs for each call that needs it and
for no other, with tuned, tile, slab and queue shapes, and in batches that replay a graph.
The reference is the oracle's processed grid."""
import numpy as np
import pytest

import oracle_api as oa

pytestmark = pytest.mark.gpu


def field(k, special):
    rng = np.random.default_rng(k)
    f = rng.uniform(-1, 1, (9, 10, 11)).astype(np.float32)
    if special:
        f[4, 5, 6], f[0, 0, 0], f[8, 9, 10] = np.float32(-0.0), np.float32(1.5e38), np.float32(np.inf)
    return f


def expect(f):
    return oa.extract(f, (0, 0, 0), (1, 1, 1), 0.25, flags=oa.PAD1, want_grid=True).grid.view(np.uint32)


@pytest.mark.parametrize("shape", [0, 2, 5, 7, 9])
def test_single(shape):
    import manifolddmc_amd as mdmc
    d = mdmc.DualMarchingCubes()
    try:
        d.set_tile_shape(shape)
        for k, special in enumerate([False, True, True, False, True, False]):
            f = field(k, special)
            print("prepare", shape, k, special, flush=True)
            d.extract_raw(f.ctypes.data, (11, 10, 9), (0, 0, 0), (1, 1, 1), 0.25, mdmc.PAD1 | mdmc.SURF_ITER)
            got = d.processed_grid()[0]
            assert np.array_equal(got.view(np.uint32), expect(f)), (shape, k)
            o = oa.extract(f, (0, 0, 0), (1, 1, 1), 0.25, flags=oa.PAD1 | oa.SURF_ITER)
            assert np.array_equal(d.mesh_numpy().halfedges, o.he)
    finally:
        d.close()


def test_batch_replays():
    import torch

    import manifolddmc_amd as mdmc
    d = mdmc.DualMarchingCubes()
    try:
        d.set_tile_shape(5)
        for k, special in enumerate([False, False, False, True, False, True]):
            fields = [field(10 * k, False), field(10 * k + 1, special)]
            t = [torch.from_numpy(f).cuda() for f in fields]
            torch.cuda.synchronize()
            print("prepare batch", k, special, flush=True)
            d.extract_batch_raw([(x.data_ptr(), (11, 10, 9), (0, 0, 0), (1, 1, 1), True) for x in t], [[0.25, 0.1]] * 2, mdmc.PAD1 | mdmc.SURF_ITER)
            for i, f in enumerate(fields):
                assert np.array_equal(d.processed_grid(i)[0].view(np.uint32), expect(f)), (k, i)
            o = oa.extract(fields[1], (0, 0, 0), (1, 1, 1), 0.25, flags=oa.PAD1 | oa.SURF_ITER)
            assert np.array_equal(d.batch_meshes()[2].halfedges, o.he), k
        assert d.graph_replays() >= 4
    finally:
        d.close()
