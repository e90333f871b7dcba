"""GPU: the FP64 discrete levels' group sizes (one node pair per wavefront up
to 64) and the classified form against the form that tests every triangle
pair (pruning off): the same contacts bit for bit."""
import numpy as np
import pytest

import delta2_amd as d2
from delta2_amd import scenes
from gpu_cases import dense_scene, hull_scene, with_future

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make", [dense_scene, hull_scene])
@pytest.mark.parametrize("copies,chunk", [(0, 1024), (1, 1024), (1, 1), (40, 1024), (40, 3)])
def test_groups_and_classification(make, copies, chunk):
    s = make()
    pairs = np.tile(s.pairs, (copies, 1)) if copies else s.pairs[:1]
    rec = with_future(s.records, scenes.DT)
    out = []
    for prune in (True, False):
        with d2.Context(0, d2.D2_FP64) as c:
            c.set_tune(chunk, 2048, 4096)
            c.set_pruning(prune)
            c.upload_trees(s.trees)
            c.upload_bodies(s.tree_of_body, rec)
            for _ in range(2):  # grids of the first run, then from its sizes
                r = d2.compare_trees_full(c, pairs, filter=False)
            out.append((r.offsets, r.ints, r.reals))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert copies == 0 or out[0][0][-1] > 0
