"""The stage times of an extraction from host memory count the field's upload, under padding and in the whole: a
PCIe 5 x16 link moves at most 64 GB/s in one direction."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 160
LINK = 64e9


@pytest.mark.parametrize("batch", [False, True])
def test_upload_is_counted(batch):
    import torch

    import manifolddmc_amd as mdmc
    t = np.linspace(-1, 1, N, dtype=np.float32)
    f = (np.sqrt(t[:, None, None] ** 2 + t[None, :, None] ** 2 + t[None, None, :] ** 2) - 0.6).astype(np.float32)
    dev = torch.from_numpy(f).cuda()
    d = mdmc.DualMarchingCubes()
    try:
        torch.cuda.synchronize()
        grid = lambda ptr, on: (ptr, (N, N, N), (-1, -1, -1), (2 / (N - 1),) * 3, on)

        def call(host):
            first = grid(f.ctypes.data, False) if host else grid(dev.data_ptr(), True)
            if batch:
                return d.extract_batch_raw([grid(dev.data_ptr(), True), first], [[0.0]] * 2, mdmc.DEFAULT_FLAGS)
            return d.extract_raw(*first[:4], 0.0, mdmc.DEFAULT_FLAGS, 0, first[4])

        least = f.nbytes / LINK * 1e3
        for rep in range(3):
            print("upload time", batch, rep, flush=True)
            a = call(True)
            assert a.ms_grid >= least and a.ms_total >= a.ms_grid, (a.ms_grid, a.ms_total, least)
            b = call(False)
            assert b.ms_grid < a.ms_grid
    finally:
        d.close()
