"""GPU: the bucket-level entry over list lengths at the edges of a wavefront's
share, a group of 64 triangle pairs and the hit scan's rounds, leaves and inner
nodes mixed: the same call one node pair at a time, byte for byte."""
import numpy as np
import pytest

import delta2_amd as d2
from delta2_amd import scenes
from gpu_cases import dense_scene, with_future

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def loaded():
    s = dense_scene()
    with d2.Context(0, d2.D2_FP64) as c:
        c.upload_trees(s.trees)
        c.upload_bodies(s.tree_of_body, with_future(s.records, scenes.DT))
        a, b = (int(v) for v in s.pairs[0])
        na, nb = (len(s.trees[s.tree_of_body[x]][0]) if not hasattr(s.trees, "offs") else
                  int(s.trees.offs[s.tree_of_body[x] + 1] - s.trees.offs[s.tree_of_body[x]]) for x in (a, b))
        rng = np.random.default_rng(3)
        kinds = np.stack([rng.integers(na, size=200), rng.integers(nb, size=200)], axis=1).astype(np.int32)
        single = [c.find_contacts_bucket(a, b, kinds[k:k + 1]) for k in range(len(kinds))]
        assert sum(r[1].shape[0] for r in single) > 0
        yield c, a, b, kinds, single


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 2049, 6007, 8192, 8193, 20000])
def test_bucket_groups(loaded, n):
    c, a, b, kinds, single = loaded
    pick = np.random.default_rng(n).integers(len(kinds), size=n)
    used, ints, reals = c.find_contacts_bucket(a, b, kinds[pick])
    assert np.array_equal(used, np.cumsum([single[k][1].shape[0] for k in pick]))
    assert np.array_equal(ints, np.concatenate([single[k][1] for k in pick]))
    assert np.array_equal(reals, np.concatenate([single[k][2] for k in pick]))
