"""A split step's passes over ranges of one launch (vertices, halfedges, faces) and its ranking of
the collapsing halfedges in tiles of 1024 corners (256 faces): random fields whose non-manifold
face counts lie below, around and above whole tiles, at every split step, against the oracle, with the
meshes growing and shrinking on one context so that grown arrays and reset maps are met again."""
import numpy as np
import pytest

import oracle_api as oa
from test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu

SPLIT = oa.SURF_ITER | oa.SPLIT_NM | oa.DETECT_NM_VERTS
SHAPES = [(3, 3, 3), (9, 9, 9), (4, 5, 6), (12, 11, 13), (7, 8, 9), (21, 20, 19), (3, 4, 3)]


@pytest.mark.parametrize("step", range(oa.STEP_NONE, oa.STEP_ITERATIVE + 1))
def test_steps(step):
    rng = np.random.default_rng(step)
    for shape in SHAPES:
        f = rng.uniform(-1, 1, shape).astype(np.float32)
        assert_same(f, (0, 0, 0), (1, 1, 1), 0.0, SPLIT | (oa.PAD1 if step & 1 else 0), split_step=step, label="%s step %d" % (shape, step))


def test_face_by_face_counts():
    """A slab of a checkerboard gains non-manifold faces cell by cell: counts through one tile's edge."""
    for n in range(2, 15):
        z, y, x = np.indices((3, n, 14))
        f = np.where((x + y + z) & 1, 1.0, -1.0).astype(np.float32)
        assert_same(f, (0, 0, 0), (1, 1, 1), 0.0, SPLIT | oa.PAD1, label="checkerboard %d" % n)
