"""A chain of simplifications whose compaction met an inconsistent quad ends in MDMC_ERR_INTERNAL, whatever stages
follow (the switch has the count raised behind the compaction, with no word to a host that went on already),
and the context then works as before."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

INTERNAL = 7


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("after", ["nothing", "split", "detect", "both"])
@pytest.mark.parametrize("chain", [("P3X3Y_COLOR",), ("P3333",), ("P3X3Y_COLOR", "P3X3Y_OLD", "P3333")])
def test_inconsistent_quad_is_reported(chain, after, batch):
    import manifolddmc_amd as mdmc
    flags = mdmc.PAD1 | mdmc.SURF_ITER
    for k in chain:
        flags |= getattr(mdmc, k)
    flags |= mdmc.SPLIT_NM if after in ("split", "both") else 0
    flags |= mdmc.DETECT_NM_VERTS if after in ("detect", "both") else 0
    f = np.random.default_rng(3).uniform(-1, 1, (14, 15, 16)).astype(np.float32)
    isos = [0.0, 0.2] if batch else [0.0]
    d = mdmc.DualMarchingCubes()
    call = lambda: d.extract_batch([f], [isos], [(0, 0, 0)], [(1, 1, 1)], flags)
    try:
        print("held chain", chain, after, batch, flush=True)
        call()
        want = d.mesh_numpy()
        d.set_fail_compaction(True)
        with pytest.raises(mdmc.MdmcError) as e:
            call()
        assert e.value.status == INTERNAL
        d.set_fail_compaction(False)
        call()
        got = d.mesh_numpy()
        assert np.array_equal(got.halfedges, want.halfedges) and np.array_equal(got.positions, want.positions)
    finally:
        d.close()


def test_switch_leaves_other_extractions_alone():
    import manifolddmc_amd as mdmc
    f = np.random.default_rng(3).uniform(-1, 1, (14, 15, 16)).astype(np.float32)
    d = mdmc.DualMarchingCubes()
    try:
        d.set_fail_compaction(True)
        st = d.extract_raw(f.ctypes.data, (16, 15, 14), (0, 0, 0), (1, 1, 1), 0.0, mdmc.DEFAULT_FLAGS)
        assert st.n_vertices > 0
    finally:
        d.close()
