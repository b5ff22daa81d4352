"""mdmc_mesh_copy into memory that the context's GPU does not own, given as device buffers: host arrays and
pinned ones (the copies serve them, as another GPU's memory), mixed with its own, shifted, batches too."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ARRAYS = ("positions", "normals", "halfedges", "face_halfedge", "face_attr", "vertex_flags", "vertex_halfedge")


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("where", ["host", "pinned", "mixed"])
def test_copy_into_other_memory(where, batch):
    import torch

    import manifolddmc_amd as mdmc
    n = 17
    f = np.random.default_rng(n).uniform(-1, 1, (n, n, n)).astype(np.float32)
    d = mdmc.DualMarchingCubes()
    try:
        d.extract_batch([f], [[0.0, 0.3] if batch else [0.0]], [(0, 0, 0)], [(1, 1, 1)], mdmc.PAD1 | mdmc.SURF_ITER | mdmc.ALL_POST)
        m = d.mesh_numpy()
        want = {k: getattr(m, k) for k in ARRAYS}
        for shift in (0, 1):
            print("copy elsewhere", where, batch, shift, flush=True)
            room, ptr = {}, {}
            for i, (k, v) in enumerate(want.items()):
                at = ("host", "pinned", "own")[i % 3] if where == "mixed" else where
                b = torch.full((v.nbytes + 64,), 0xA5, dtype=torch.uint8, device="cuda" if at == "own" else "cpu", pin_memory=at == "pinned")
                room[k], ptr[k] = b, b.data_ptr() + shift * v.dtype.itemsize
            torch.cuda.synchronize()
            d.copy_device(**ptr)
            for k, v in want.items():
                b = room[k].cpu().numpy()
                o = shift * v.dtype.itemsize
                assert np.array_equal(b[o:o + v.nbytes].view(v.dtype).reshape(v.shape), v), k
                assert (b[:o] == 0xA5).all() and (b[o + v.nbytes:] == 0xA5).all(), k
    finally:
        d.close()
