"""GPU: the FP32 form's mask kernel over list sizes that end inside a
wavefront, a group of 64 triangles and a block's tile, with and without
pruning: the FP64 form's contacts bit for bit."""
import numpy as np
import pytest

import delta2_amd as d2
from delta2_amd import scenes
from gpu_cases import dense_scene, hull_scene, with_future

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make", [dense_scene, hull_scene])
@pytest.mark.parametrize("copies,chunk", [(0, 1024), (1, 1024), (1, 1), (7, 2), (60, 1024)])
def test_mask_groups(make, copies, chunk):
    s = make()
    pairs = np.tile(s.pairs, (copies, 1)) if copies else s.pairs[:1]
    rec = with_future(s.records, scenes.DT)
    out = []
    for precision, prune in ((d2.D2_FP64, True), (d2.D2_FP32, True), (d2.D2_FP32, False)):
        with d2.Context(0, precision) as c:
            c.set_tune(chunk, 2048, 4096)
            c.set_pruning(prune)
            c.upload_trees(s.trees)
            c.upload_bodies(s.tree_of_body, rec)
            for _ in range(2):  # grids of the first run, then from its sizes
                r = d2.compare_trees_full(c, pairs, filter=False)
            out.append((r.offsets, r.ints, r.reals))
    for b in out[1:]:
        for x, y in zip(out[0], b):
            assert np.array_equal(x, y)
    assert copies == 0 or out[0][0][-1] > 0
