"""GPU: the pair certificate's two forms -- a wavefront per pair for hulls of up
to 256 vertices, a block above -- over pair counts that end inside a block, on
scenes that hold both kinds: every pair is proposed and counted once, some are
certified, and the runs return exactly the ungated results."""
import numpy as np
import pytest

import delta2_amd as d2
from delta2_amd import scenes
from gpu_cases import hull_scene, sparse_scene
from test_gpu_learned import propose_all

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make,copies", [(sparse_scene, 1), (sparse_scene, 12), (hull_scene, 1), (hull_scene, 3)])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 61, None])
def test_certificate_forms(make, copies, n):
    s = make()
    pairs = np.tile(s.pairs, (copies, 1))[:n]
    mt = np.full(pairs.shape[0], scenes.DT)
    out = []
    for gated in (False, True):
        with d2.Context(0, d2.D2_FP32) as c:
            if gated:
                c.mlp_set_params(propose_all())
            c.set_learned(gated)
            c.upload_trees(s.trees)
            c.upload_bodies(s.tree_of_body, s.records)
            for _ in range(2):
                r = d2.compare_trees_full_continuous(c, pairs, mt)
            out.append((r.offsets, r.ints, r.reals, r.per_pair))
            if gated:
                proposed, certified = c.gate_counts()["ccd"]
                assert proposed == pairs.shape[0] and 0 <= certified <= proposed
                assert n is not None or make is not sparse_scene or certified > 0
    for x, y in zip(*out):
        assert np.array_equal(x, y)
