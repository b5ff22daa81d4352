"""A batch's regroup: every problem's arrays, offsets, statistics and DMC counts equal those of its
own extraction -- with and without a split (nothing to move without one), a fixture that splits
twice between others (tails of several runs), empty problems first, last and in between, statistics
chunks holding many problems and problems holding many chunks, tile, slab and queue shapes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def fields():
    rng = np.random.default_rng(5)
    flat = np.ones((3, 4, 5), np.float32)
    tiny = [rng.uniform(-1, 1, (3, 3, 3)).astype(np.float32) for _ in range(40)]
    noisy = [rng.uniform(-1, 1, (n, n + 1, n + 2)).astype(np.float32) for n in (6, 13, 21)]
    x = np.linspace(-1, 1, 40, dtype=np.float32)
    ball = (np.sqrt(x[:, None, None] ** 2 + x[None, :, None] ** 2 + x[None, None, :] ** 2) - 0.7).astype(np.float32)
    return [flat] + tiny[:20] + [ball, noisy[0], flat] + tiny[20:] + noisy[1:] + [flat]


FLAG_SETS = {"dual": "PAD1 SURF_ITER", "detect": "SURF_ITER DETECT_NM_VERTS", "default": "PAD1 SURF_ITER SPLIT_NM DETECT_NM_VERTS",
             "chain": "PAD1 SURF_ITER P3X3Y_COLOR P3333", "all": "PAD1 SURF_ITER P3X3Y_COLOR P3X3Y_OLD P3333 SPLIT_NM DETECT_NM_VERTS",
             "all_unpadded": "SURF_ITER P3X3Y_COLOR P3X3Y_OLD P3333 SPLIT_NM DETECT_NM_VERTS"}


@pytest.mark.parametrize("shape,flags_name", [(0, k) for k in FLAG_SETS] + [(2, "all"), (5, "default"), (7, "all"), (8, "default"), (9, "all")])
def test_problems_equal_their_own_extractions(shape, flags_name):
    import manifolddmc_amd as mdmc
    flags = 0
    for k in FLAG_SETS[flags_name].split():
        flags |= getattr(mdmc, k)
    fs = fields()
    isos = [[0.0, 0.35]] * len(fs)
    o, dl = (0.0, 0.0, 0.0), (1.0, 1.0, 1.0)
    d, one = mdmc.DualMarchingCubes(), mdmc.DualMarchingCubes()
    try:
        d.set_tile_shape(shape)
        for repeat in range(2):
            print("regroup", shape, flags_name, repeat, flush=True)
            st = d.extract_batch(fs, isos, [o] * len(fs), [dl] * len(fs), flags)
            meshes, stats = d.batch_meshes(), d.batch_stats()
        worst = 0
        for i, f in enumerate(fs):
            for k, iso in enumerate(isos[i]):
                b = 2 * i + k
                s = one.extract_raw(f.ctypes.data, f.shape[::-1], o, dl, iso, flags)
                worst = max(worst, s.split_iterations)
                m = one.mesh_numpy()
                for name in ("positions", "normals", "halfedges", "face_halfedge", "face_attr", "vertex_flags", "vertex_halfedge"):
                    assert np.array_equal(getattr(meshes[b], name), getattr(m, name)), (b, name)
                for name in ("n_vertices", "n_halfedges", "n_faces", "n_dmc_vertices", "n_dmc_quads", "nm_edges4", "nm_edges3", "n_edges", "nm_vertices"):
                    assert getattr(stats[b], name) == getattr(s, name), (b, name)
                assert list(stats[b].quads_with_nm) == list(s.quads_with_nm), b
        assert worst == st.split_iterations
    finally:
        d.close()
        one.close()


@pytest.mark.parametrize("flags_name", ["default", "all"])
def test_several_split_iterations(flags_name):
    import fixtures
    import manifolddmc_amd as mdmc
    flags = 0
    for k in FLAG_SETS[flags_name].split():
        flags |= getattr(mdmc, k)
    vals, origin, delta, iso = fixtures.load_problem("Iterative-Fix")
    vals = np.ascontiguousarray(vals, np.float32)
    rng = np.random.default_rng(2)
    noisy = rng.uniform(iso - 1, iso + 1, (9, 8, 7)).astype(np.float32)
    fs = [vals, noisy, vals, vals, noisy, vals]
    d, one = mdmc.DualMarchingCubes(), mdmc.DualMarchingCubes()
    try:
        st = d.extract_batch(fs, [[iso]] * len(fs), [origin] * len(fs), [delta] * len(fs), flags)
        assert st.split_iterations >= 2
        for b, (f, g) in enumerate(zip(fs, d.batch_meshes())):
            one.extract_raw(f.ctypes.data, f.shape[::-1], origin, delta, iso, flags)
            m = one.mesh_numpy()
            for name in ("positions", "normals", "halfedges", "face_halfedge", "face_attr", "vertex_flags", "vertex_halfedge"):
                assert np.array_equal(getattr(g, name), getattr(m, name)), (b, name)
    finally:
        d.close()
        one.close()
