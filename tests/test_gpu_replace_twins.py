"""P3333 merges whose centre takes over the outer halfedges of its removed neighbours (twins replaced,
no list searched) against the oracle and against the rebuild of everything around the targets
(mdmc_set_local_merges(0)): smooth meshes with many regular centres, some next to each other, sharing
targets or at the border, and noisy ones with buckets of three and more around them; P3333 alone and
after the other simplifications."""
import numpy as np
import pytest

import oracle_api as oa
from test_gpu_parity import assert_same
from test_gpu_simplify_chain import extract

pytestmark = pytest.mark.gpu


def waves(shape, noise, seed):
    rng = np.random.default_rng(seed)
    z, y, x = np.meshgrid(*[np.arange(n, dtype=np.float32) for n in shape], indexing="ij")
    f = np.sin(0.7 * x) * np.cos(0.6 * y) + np.sin(0.65 * y) * np.cos(0.7 * z) + np.sin(0.6 * z) * np.cos(0.65 * x)
    return (f + noise * rng.uniform(-1, 1, shape)).astype(np.float32)


@pytest.mark.parametrize("noise", [0.0, 0.05, 0.2, 0.6])
@pytest.mark.parametrize("pre", [0, oa.P3X3Y_COLOR, oa.P3X3Y_OLD, oa.P3X3Y_COLOR | oa.P3X3Y_OLD])
def test_against_oracle_and_rebuild(noise, pre):
    for k, shape in enumerate([(30, 31, 33), (5, 40, 40), (40, 6, 7), (48, 48, 48)]):
        f = waves(shape, noise, 10 * k + 1)
        for pad in (0, oa.PAD1):
            flags = pad | pre | oa.P3333
            assert_same(f, (0, 0, 0), (1, 1, 1), 0.1, flags, label="noise %g %s" % (noise, shape))
            a, _ = extract(f, 0.1, flags, True)
            b, _ = extract(f, 0.1, flags, False)
            for name in ("halfedges", "face_halfedge", "face_attr", "vertex_flags", "vertex_halfedge", "positions"):
                assert np.array_equal(getattr(a, name), getattr(b, name)), (noise, shape, name)
