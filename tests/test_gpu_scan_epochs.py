"""The prefix sums' look-back words are told apart by a 16-bit launch epoch instead of being
cleared: meshes stay the same while the epochs run out and start again, with scans of one and
of several tiles in between."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_epochs_wrap():
    import torch

    import manifolddmc_amd as mdmc
    rng = np.random.default_rng(3)
    small = torch.from_numpy(rng.uniform(-1, 1, (3, 4, 3)).astype(np.float32)).cuda()
    large = torch.from_numpy(rng.uniform(-1, 1, (26, 26, 26)).astype(np.float32)).cuda()
    torch.cuda.synchronize()
    d = mdmc.DualMarchingCubes()

    def run(t):
        nz, ny, nx = t.shape
        st = d.extract_raw(t.data_ptr(), (nx, ny, nz), (0, 0, 0), (1, 1, 1), 0.0, mdmc.PAD1, 0, True)
        assert st.lookback_fallbacks == 0
        return st

    try:
        run(large)  # more than 8 tiles of 4096 vertices
        want = d.mesh_numpy()
        assert len(want.positions) > 8 * 4096 // 2
        for k in range(66000):  # at least one epoch per extraction
            run(small)
            if k % 3000 == 0 or k > 65400 and k % 40 == 0:
                print("extraction", k, flush=True)
                run(large)
                got = d.mesh_numpy()
                assert np.array_equal(got.halfedges, want.halfedges) and np.array_equal(got.positions, want.positions)
    finally:
        d.close()
