"""mdmc_mesh_quads: the faces' vertex ids and the positions of one launch equal those of the
copied mesh, on an empty mesh, sizes around a block's edges and a mesh the splitter rewrote."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,flags_name", [(2, "DEFAULT_FLAGS"), (5, "DEFAULT_FLAGS"), (9, "RECORD"), (24, "DEFAULT_FLAGS"), (24, "ALL")])
def test_quads_equal_mesh_copy(n, flags_name):
    import torch

    import manifolddmc_amd as mdmc
    flags = {"DEFAULT_FLAGS": mdmc.DEFAULT_FLAGS, "RECORD": mdmc.PAD1 | mdmc.RECORD_ADJOINT, "ALL": mdmc.PAD1 | mdmc.SURF_ITER | mdmc.ALL_POST}[flags_name]
    rng = np.random.default_rng(n)
    f = rng.uniform(-1, 1, (n, n, n)).astype(np.float32) if n > 2 else np.ones((n, n, n), np.float32)
    d = mdmc.DualMarchingCubes()
    try:
        t = torch.from_numpy(f).cuda()
        torch.cuda.synchronize()
        d.extract_raw(t.data_ptr(), (n, n, n), (0, 0, 0), (1, 1, 1), 0.0, flags, 0, True)
        V, H, F = d.info()
        m = d.mesh_numpy()
        assert (V > 0) == (n > 2)
        pos = torch.full((V + 1, 3), 7.0, device="cuda")
        room = torch.full((4 * F + 3,), -7, dtype=torch.int64, device="cuda")
        for shift in (0, 1):  # 16-byte aligned ids, and not
            torch.cuda.synchronize()
            d.copy_quads(pos.data_ptr(), room.data_ptr() + 8 * shift)
            torch.cuda.synchronize()
            q = room[shift:shift + 4 * F].reshape(F, 4).cpu().numpy()
            assert np.array_equal(q, m.faces().astype(np.int64))
            assert int(room[shift + 4 * F]) == -7
        assert np.array_equal(pos[:V].cpu().numpy(), m.positions) and bool((pos[V] == 7.0).all())
    finally:
        d.close()
