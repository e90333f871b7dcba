"""GPU: a graph captured with the learned gate on, then another tree set with
the same body, pair and level counts that fits the buffers already there.  The
certificate has a second launch for hulls of more than 256 vertices, so a graph
of small hulls does not serve a set that holds larger ones, nor the reverse:
the runs after the upload propose every pair and return an ungated context's
results."""
import numpy as np
import pytest

import delta2_amd as d2
from delta2_amd import pcg_seed, scenes
from test_gpu_learned import propose_all

pytestmark = pytest.mark.gpu
N = 40
PAIRS = np.array([(i, j) for i in range(N) for j in range(i + 1, N)], dtype=np.int32)


def hull_trees(points, depth=3):
    """Trees of the given depth, one per entry: the hull of that many points on
    the unit sphere (all of them vertices)."""
    out = []
    for k, n in enumerate(points):
        for seed in range(100 * k, 100 * k + 100):
            d = np.random.default_rng(seed).normal(size=(n, 3))
            V, F = scenes.convex_hull_mesh(d / np.linalg.norm(d, axis=1, keepdims=True))
            tree = scenes.tree_build(V, F, pcg_seed(42, seed))
            if len(V) == n and tree[0][:, 3].max() == depth:
                out.append(tree)
                break
    assert len(out) == len(points)
    return out


def records():
    rng = np.random.default_rng(4)
    pos = rng.uniform(0.0, 5.0, size=(N, 3))
    return np.stack([scenes.body_record(np.array([1.0, 0, 0, 0]), p, rng.normal(0, 1.0, size=3), np.eye(3)) for p in pos])


def load(c, trees, rec):
    c.upload_trees(trees)
    c.upload_bodies(np.arange(N, dtype=np.int32) % len(trees), rec)
    c.upload_pairs(PAIRS, np.full(PAIRS.shape[0], scenes.DT))


def results(c, op):
    c.ccd_run() if op == "ccd" else c.narrow_run(True)
    r = c.result(with_pairs=op == "ccd")
    return r.offsets, r.ints, r.reals


@pytest.mark.parametrize("op", ["ccd", "discrete"])
@pytest.mark.parametrize("order", ["small first", "large first"])
def test_tree_set_with_larger_hulls_after_capture(op, order):
    small, large = hull_trees([240] * 14), hull_trees([160, 160, 160, 260, 160, 270])
    sets = [small, large, small] if order == "small first" else [small, large, large, small, large]
    rec = records()
    with d2.Context(0, d2.D2_FP32) as g, d2.Context(0, d2.D2_FP32) as plain:
        g.mlp_set_params(propose_all())
        g.set_learned(True)
        g.set_graph(True)
        for trees in sets:
            load(plain, trees, rec)
            want = results(plain, op)
            assert want[0][-1] > 100
            load(g, trees, rec)
            for k in range(3):
                got = results(g, op)
                proposed, certified = g.gate_counts()["ccd" if op == "ccd" else "discrete"]
                assert proposed == PAIRS.shape[0] and 0 < certified < proposed, (k, proposed, certified)
                for x, y in zip(got, want):
                    assert np.array_equal(x, y), k
        assert g.graph_stats()[1] > 0
