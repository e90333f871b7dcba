"""GPU: the CCD levels' lists over sizes that end inside a wavefront, a group
of 64 triangles or vertices, a block's tile and the survivor buffers (one block
for everything), FP32 culls against the FP64 form: the same contacts and
minimum times bit for bit."""
import numpy as np
import pytest

import delta2_amd as d2
from delta2_amd import scenes
from gpu_cases import dense_scene, hull_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make", [dense_scene, hull_scene])
@pytest.mark.parametrize("copies,chunk,stream", [(0, 1024, 2048), (1, 1024, 2048), (1, 1, 1), (7, 2, 3), (40, 1024, 2048)])
def test_ccd_lists(make, copies, chunk, stream):
    s = make()
    pairs = np.tile(s.pairs, (copies, 1)) if copies else s.pairs[:1]
    mt = np.full(pairs.shape[0], 4 * scenes.DT)
    out = []
    for precision in (d2.D2_FP64, d2.D2_FP32):
        with d2.Context(0, precision) as c:
            c.set_tune(chunk, stream, 4096)
            c.upload_trees(s.trees)
            c.upload_bodies(s.tree_of_body, s.records)
            for _ in range(2):  # grids of the first run, then from its sizes
                r = d2.compare_trees_full_continuous(c, pairs, mt)
                out.append((r.offsets, r.ints, r.reals, r.per_pair))
    for b in out[1:]:
        for x, y in zip(out[0], b):
            assert np.array_equal(x, y)
    assert copies == 0 or out[0][0][-1] > 0
