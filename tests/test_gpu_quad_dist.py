"""GPU: the triangle test by four lanes against the one by a lane: the same
discrete contacts bit for bit, on lists below and above the bound between the
two and through it from one run to the next."""
import numpy as np
import pytest

import delta2_amd as d2
from delta2_amd import scenes
from gpu_cases import dense_scene, hull_scene, with_future

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make", [dense_scene, hull_scene])
@pytest.mark.parametrize("copies", [0, 1, 3, 30])
def test_quads_and_lanes_agree(make, copies):
    s = make()
    pairs = np.tile(s.pairs, (copies, 1)) if copies else s.pairs[:1]
    rec = with_future(s.records, scenes.DT)
    with d2.Context(0, d2.D2_FP64) as c:  # one lane per test
        c.upload_trees(s.trees)
        c.upload_bodies(s.tree_of_body, rec)
        want = d2.compare_trees_full(c, pairs, filter=False)
    with d2.Context(0, d2.D2_FP32) as c:  # the first run has no sizes to go by: one lane; then by size
        c.upload_trees(s.trees)
        c.upload_bodies(s.tree_of_body, rec)
        for _ in range(3):
            got = d2.compare_trees_full(c, pairs, filter=False)
            for x, y in ((want.offsets, got.offsets), (want.ints, got.ints), (want.reals, got.reals)):
                assert np.array_equal(x, y)
