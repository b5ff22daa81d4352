"""The initialize finds a halfedge's bucket from its vertices' contours where the cells' common face
has two crossed edges or two neighbouring ones of four, and searches the vertex lists for the
rest: every sign pattern of two neighbouring cells along each axis (random +-1 fields, whose ties
the decider breaks, and uniform noise), at the grid's border and inside, with one and two cells
across, both with the records built at once and with a simplification before them, against the
oracle."""
import numpy as np
import pytest

import oracle_api as oa
from test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu


def noise(kind, shape, seed):
    rng = np.random.default_rng(seed)
    if kind == "sign":
        return rng.choice([-1.0, 1.0], shape).astype(np.float32)
    return rng.uniform(-1, 1, shape).astype(np.float32)


@pytest.mark.parametrize("kind", ["sign", "uniform"])
@pytest.mark.parametrize("flags", [0, oa.PAD1 | oa.SURF_ITER, oa.P3X3Y_COLOR, oa.PAD1 | oa.P3X3Y_COLOR | oa.P3X3Y_OLD | oa.P3333])
def test_sign_patterns(kind, flags):
    for k, shape in enumerate([(21, 22, 20), (2, 2, 2), (2, 9, 9), (9, 2, 9), (9, 9, 2), (3, 3, 17), (17, 3, 3), (3, 17, 3)]):
        assert_same(noise(kind, shape, 100 + k), (0, 0, 0), (1, 1, 1), 0.0, flags, label="%s %s" % (kind, shape))


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_two_cells_every_pattern(axis):
    """Blocks of 3 x 2 x 2 samples with all 4096 sign patterns, kept apart by one positive layer."""
    n = 4096
    f = np.ones((4, 3 * 64, 3 * 64), np.float32)
    bits = ((np.arange(n)[:, None] >> np.arange(12)) & 1).astype(np.float32) * -2 + 1
    for p in range(n):
        y, x = divmod(p, 64)
        f[:3, 3 * y:3 * y + 2, 3 * x:3 * x + 2] = bits[p].reshape(3, 2, 2)
    f = np.ascontiguousarray(np.moveaxis(f, 0, axis))
    for flags in (oa.PAD1, oa.PAD1 | oa.P3333):
        assert_same(f, (0, 0, 0), (1, 1, 1), 0.0, flags, label="axis %d" % axis)
