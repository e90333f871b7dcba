"""GPU: the profiling counters describe the launches they stand beside: the
items of every kernel that launched are the sum over the run's levels of what
those launches took, and a kernel that takes no part in a run shows no time."""
import numpy as np
import pytest

import delta2_amd as d2
from delta2_amd import scenes
from gpu_cases import dense_scene, with_future

pytestmark = pytest.mark.gpu
SOUP, CONN, ITEMS, PT, EE, SPT, SEE = range(7)  # a level's sizes


@pytest.mark.parametrize("prec", [d2.D2_FP64, d2.D2_FP32], ids=["fp64", "fp32"])
def test_ccd_items_per_launch(prec):
    s = dense_scene()
    with d2.Context(0, prec) as c:
        c.upload_trees(s.trees)
        c.upload_bodies(s.tree_of_body, s.records)
        c.set_profiling(True)
        d2.compare_trees_full_continuous(c, s.pairs, np.full(s.pairs.shape[0], 4 * scenes.DT))
        st = c.kernel_stats()
        lv = c.run_info()[1][0].sum(axis=0)  # ([1] keeps the phase's contact count in its last field)
    soup_sub = lv[SPT] + lv[SEE] if prec == d2.D2_FP32 else 15 * lv[ITEMS]
    want = {"soup_cull": lv[SOUP] + lv[CONN], "soup_edge": soup_sub + lv[PT] + lv[EE], "soup_reduce": lv[ITEMS]}
    if prec == d2.D2_FP32:
        want["soup_keep"] = lv[ITEMS]
    assert lv[ITEMS] > 0 and lv[CONN] > 0
    for k, n in want.items():
        assert st[k][0] > 0 and st[k][2] == n, (k, st[k], n)
    assert st["leaf_point"][2] == lv[PT] and st["leaf_edge"][2] == lv[EE]
    for k in ("soup_point", "leaf_point", "leaf_edge"):
        assert st[k][0] == 0 and st[k][1] == 0.0, k
    assert st["expand"] == (0, 0.0, 0.0)


@pytest.mark.parametrize("prec", [d2.D2_FP64, d2.D2_FP32], ids=["fp64", "fp32"])
def test_discrete_items_per_launch(prec):
    s = dense_scene()
    with d2.Context(0, prec) as c:
        c.upload_trees(s.trees)
        c.upload_bodies(s.tree_of_body, with_future(s.records, scenes.DT))
        c.set_profiling(True)
        d2.compare_trees_full(c, s.pairs, filter=False)
        st = c.kernel_stats()
        lv = c.run_info()[1][0].sum(axis=0)
    if prec == d2.D2_FP32:
        want = {"tri_mask": lv[SOUP], "tri_dist": lv[ITEMS]}
        assert st["expand"] == (0, 0.0, 0.0) and st["tri_full"] == (0, 0.0, 0.0)
    else:
        want = {"tri_full": lv[ITEMS], "expand": lv[SOUP]}
    for k, n in want.items():
        assert st[k][0] > 0 and st[k][2] == n, (k, st[k], n)
