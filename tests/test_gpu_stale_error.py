"""An error that an earlier HIP call of the thread left behind (here a device number that does not exist)
is none of the extraction's: single and batched calls, empty ones, and every copy of the mesh work as ever."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def leave_error():
    name = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    hip = ctypes.CDLL(name)
    assert hip.hipSetDevice(1 << 20) != 0
    return hip


@pytest.mark.parametrize("flags_name", ["DEFAULT_FLAGS", "ALL"])
def test_an_earlier_error_is_not_the_extractions(flags_name):
    import torch

    import manifolddmc_amd as mdmc
    flags = {"DEFAULT_FLAGS": mdmc.DEFAULT_FLAGS, "ALL": mdmc.PAD1 | mdmc.SURF_ITER | mdmc.ALL_POST}[flags_name]
    f = np.random.default_rng(4).uniform(-1, 1, (12, 13, 14)).astype(np.float32)
    empty = np.ones((5, 5, 5), np.float32)
    dims, empty_dims = (14, 13, 12), (5, 5, 5)
    d = mdmc.DualMarchingCubes()
    try:
        d.extract_raw(f.ctypes.data, dims, (0, 0, 0), (1, 1, 1), 0.0, flags)
        want = d.mesh_numpy()
        pos = torch.zeros(want.positions.shape, device="cuda")
        quads = torch.zeros((len(want.face_halfedge), 4), dtype=torch.int64, device="cuda")
        again = torch.zeros_like(pos)
        torch.cuda.synchronize()
        hip = leave_error()
        d.extract_raw(f.ctypes.data, dims, (0, 0, 0), (1, 1, 1), 0.0, flags)
        leave_error()
        got = d.mesh_numpy()
        leave_error()
        d.copy_device(positions=pos.data_ptr())
        leave_error()
        d.copy_quads(again.data_ptr(), quads.data_ptr())
        leave_error()
        d.extract_raw(empty.ctypes.data, empty_dims, (0, 0, 0), (1, 1, 1), 0.0, flags)
        none = d.info()
        leave_error()
        d.extract_batch([f, empty], [[0.0], [0.0]], [(0, 0, 0)] * 2, [(1, 1, 1)] * 2, flags)
        first = d.batch_meshes()[0]
        hip.hipGetLastError()  # torch would report it
        assert np.array_equal(got.halfedges, want.halfedges) and np.array_equal(got.positions, want.positions)
        assert np.array_equal(pos.cpu().numpy(), want.positions) and np.array_equal(again.cpu().numpy(), want.positions)
        he, at = want.halfedges, want.face_halfedge
        for k in range(4):
            assert np.array_equal(quads[:, k].cpu().numpy(), he[at, 0])
            at = he[at, 2]
        assert none == (0, 0, 0)
        assert np.array_equal(first.halfedges, want.halfedges)
    finally:
        d.close()
