"""The last stages launched behind the non-manifold face list without waiting for it: nothing to
split, iterations cut short (faces left when detection and statistics run), single split
steps, vertices left to the slow fan pass, detection off -- arrays and counts as the oracle's,
extraction after extraction on one context."""
import numpy as np
import pytest

import fixtures
import oracle_api as oa
from test_gpu_parity import assert_same, gpu

pytestmark = pytest.mark.gpu


def fields():
    rng = np.random.default_rng(7)
    noisy = rng.uniform(-1, 1, (11, 12, 13)).astype(np.float32)
    x = np.linspace(-1, 1, 20, dtype=np.float32)
    ball = (x[:, None, None] ** 2 + x[None, :, None] ** 2 + x[None, None, :] ** 2 - 0.5).astype(np.float32)
    return {"noisy": (noisy, 0.1), "ball": (ball, 0.0), "flat": (np.ones((3, 3, 3), np.float32), 2.0)}


@pytest.mark.parametrize("pad", [0, oa.PAD1])
@pytest.mark.parametrize("stage", ["dual", "detect", "split", "split_detect"])
def test_stages(stage, pad):
    fl = pad | {"dual": 0, "detect": oa.DETECT_NM_VERTS, "split": oa.SPLIT_NM, "split_detect": oa.SPLIT_NM | oa.DETECT_NM_VERTS}[stage]
    for name, (f, iso) in fields().items():
        for more in (oa.SURF_ITER, oa.SURF_ITER | oa.P3X3Y_COLOR, oa.P3333):
            for step in (oa.STEP_ALL, oa.STEP_SUBDIVIDE, oa.STEP_TWINS) if fl & oa.SPLIT_NM else (oa.STEP_ALL,):
                assert_same(f, (0, 0, 0), (1, 1, 1), iso, fl | more, split_step=step, label="%s %s step %d" % (name, stage, step))


@pytest.mark.parametrize("iters", [1, 2])
def test_iterations_cut_short(iters):
    d = gpu()
    rng = np.random.default_rng(1)
    cases = [fixtures.load_problem("Iterative-Fix"), (rng.uniform(-1, 1, (14, 13, 12)).astype(np.float32), (0, 0, 0), (1, 1, 1), 0.0)]
    for vals, origin, delta, iso in cases:
        flags = oa.SURF_ITER | oa.PAD1 | oa.SPLIT_NM | oa.DETECT_NM_VERTS
        d.splitting_step, d.max_split_iterations = oa.STEP_ALL, iters
        try:
            v = np.ascontiguousarray(vals, np.float32)
            st = d.extract_raw(v.ctypes.data, v.shape[::-1], origin, delta, iso, flags).as_dict()
            m = d.mesh_numpy()
        finally:
            d.max_split_iterations = 64
        o = oa.extract(vals, origin, delta, iso, flags=flags, max_split_iters=iters)
        assert np.array_equal(m.halfedges, o.he) and np.array_equal(m.vertex_flags, o.vflags)
        for k in ("nm_edges4", "nm_edges3", "n_edges", "nm_vertices", "quads_with_nm", "split_iterations", "anomalies"):
            assert st[k] == o.stats[k], k
