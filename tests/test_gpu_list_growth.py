"""GPU: work lists too short for a scene: refused while growth is off, with
nothing written past them, and grown on demand to the same results (a CCD level
of the FP32 form keeps fewer sub-tests than it has soup items, so the lists grow
to different lengths)."""
import numpy as np
import pytest

import delta2_amd as d2
from delta2_amd import scenes
from gpu_cases import dense_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [d2.D2_FP64, d2.D2_FP32])
def test_ccd_lists_at_their_limit(precision):
    """Lists too short for the scene: refused when growth is off, and nothing
    written past them; the same results once they are long enough."""
    s = dense_scene()
    pairs = np.tile(s.pairs, (4, 1))
    mt = np.full(pairs.shape[0], 4 * scenes.DT)
    with d2.Context(0, precision) as c:
        c.upload_trees(s.trees)
        c.upload_bodies(s.tree_of_body, s.records)
        want = d2.compare_trees_full_continuous(c, pairs, mt)
    with d2.Context(0, precision) as c:
        c.upload_trees(s.trees)
        c.upload_bodies(s.tree_of_body, s.records)
        c.set_capacity(pairs.shape[0] + 1)
        with pytest.raises(d2.CapacityError):
            d2.compare_trees_full_continuous(c, pairs, mt)
        c.set_auto_grow(True)
        got = d2.compare_trees_full_continuous(c, pairs, mt)
    for x, y in ((want.offsets, got.offsets), (want.ints, got.ints), (want.reals, got.reals), (want.per_pair, got.per_pair)):
        assert np.array_equal(x, y)
