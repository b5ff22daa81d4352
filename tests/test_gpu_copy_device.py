"""mdmc_mesh_copy into device buffers against the copy into host arrays: aligned and shifted
buffers, meshes smaller and larger than a block's share, with split additions, batches, and
nothing written past an array's end."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,flags_name,batch", [(2, "DEFAULT_FLAGS", False), (4, "DEFAULT_FLAGS", False), (13, "ALL", False), (40, "ALL", False),
                                                (40, "DUAL", False), (21, "DEFAULT_FLAGS", True)])
@pytest.mark.parametrize("shift", [0, 1])
def test_device_copy_equals_host_copy(n, flags_name, batch, shift):
    import torch

    import manifolddmc_amd as mdmc
    flags = {"DEFAULT_FLAGS": mdmc.DEFAULT_FLAGS, "DUAL": mdmc.PAD1 | mdmc.SURF_ITER, "ALL": mdmc.PAD1 | mdmc.SURF_ITER | mdmc.ALL_POST}[flags_name]
    rng = np.random.default_rng(n)
    f = rng.uniform(-1, 1, (n, n, n)).astype(np.float32) if n > 2 else np.ones((n, n, n), np.float32)
    d = mdmc.DualMarchingCubes()
    try:
        t = torch.from_numpy(f).cuda()
        torch.cuda.synchronize()
        print("device copy", n, flags_name, batch, shift, flush=True)
        if batch:
            d.extract_batch_raw([(t.data_ptr(), (n, n, n), (0, 0, 0), (1, 1, 1), True)], [[0.0, 0.3]], flags)
        else:
            d.extract_raw(t.data_ptr(), (n, n, n), (0, 0, 0), (1, 1, 1), 0.0, flags, 0, True)
        V, H, F = d.info()
        m = d.mesh_numpy()
        want = {"positions": m.positions, "normals": m.normals, "halfedges": m.halfedges, "face_halfedge": m.face_halfedge, "face_attr": m.face_attr,
                "vertex_flags": m.vertex_flags, "vertex_halfedge": m.vertex_halfedge}
        room = {k: torch.full((v.nbytes + 64,), 0xA5, dtype=torch.uint8, device="cuda") for k, v in want.items()}
        torch.cuda.synchronize()
        d.copy_device(**{k: b.data_ptr() + shift * want[k].dtype.itemsize for k, b in room.items()})
        for k, v in want.items():
            b = room[k].cpu().numpy()
            o = shift * v.dtype.itemsize
            assert np.array_equal(b[o:o + v.nbytes].view(v.dtype).reshape(v.shape), v), k
            assert (b[:o] == 0xA5).all() and (b[o + v.nbytes:] == 0xA5).all(), k
    finally:
        d.close()
