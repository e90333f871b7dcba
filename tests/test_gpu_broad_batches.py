"""GPU: the broad phase's item batches at their edges -- fewer bodies than one
wavefront's batch, a ragged last group, partner lists that overflow a
wavefront's shared LDS room one after another (each below its capacity), and a
static body's segments -- and cluster separation of one chain, one blob and
scattered bodies.  Pair lists and clusters equal the oracle's, as integers."""
import numpy as np
import pytest

import d2o
import delta2_amd as d2
from broad_cases import CUBE_F, CUBE_V, particle
from delta2_amd import pcg_seed, tree_build

pytestmark = pytest.mark.gpu


def check(records):
    n = records.shape[0]
    box, rad = d2o.mesh_bounds(CUBE_V)
    with d2.Context(0, d2.D2_FP64) as c:
        c.upload_trees([tree_build(CUBE_V, CUBE_F, pcg_seed(42, 54))])
        c.upload_bodies(np.zeros(n, dtype=np.int32), records)
        c.broad_phase(mode=0, t=0.01)
        pairs, _ = c.download_pairs()
        k = c.build_clusters()
        cl = c.download_clusters()
    want = d2o.broad_phase(records, np.tile(box, (n, 1)), np.full(n, rad), mode=0, t=0.01)
    assert np.array_equal(pairs, want)
    # components of the dynamic-dynamic pairs, numbered by smallest member
    root = np.arange(n)

    def find(x):
        while root[x] != x:
            root[x] = root[root[x]]
            x = root[x]
        return x

    static = records[:, 38] != 0
    for a, b in want:
        if not static[a] and not static[b]:
            ra, rb = find(a), find(b)
            root[max(ra, rb)] = min(ra, rb)
    lab = np.array([find(i) for i in range(n)])
    firsts = np.unique(lab[~static])
    assert k == firsts.size and np.array_equal(cl["first"], firsts)
    assert np.array_equal(cl["of_body"], np.where(static, -1, np.searchsorted(firsts, lab)))
    return pairs.shape[0]


@pytest.mark.parametrize("n", [1, 7, 8, 9, 31, 32, 33, 257])
def test_chain(n):
    rng = np.random.default_rng(n)
    order = rng.permutation(n)  # neighbours are 3 m apart, their spheres overlap; indices in random order
    assert check(np.stack([particle(pos=(3.0 * order[i], 0, 0)) for i in range(n)])) == n - 1


@pytest.mark.parametrize("n,n_static", [(150, 0), (400, 0), (700, 0), (1200, 3)])
def test_blob(n, n_static):
    rng = np.random.default_rng(n)
    rec = np.stack([particle(pos=rng.uniform(0, 2.0, size=3), static=i % 400 == 1 and n_static > i // 400)
                    for i in range(n)])
    assert check(rec) >= n * (n - 1) // 2 - 3 * n_static


def test_scattered():
    rng = np.random.default_rng(5)
    check(np.stack([particle(pos=rng.uniform(0, 60.0, size=3), static=i in (0, 1777)) for i in range(3000)]))
