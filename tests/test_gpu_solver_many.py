"""GPU: the solver over thousands of small clusters, which a lane each solves,
among larger ones that a block each solves: single spheres on one floor or on
two coplanar ones, stacks of two and 2 x 2 layers, in either body order, against
the oracle's sequential walk over two steps.  The comparison and its 1e-9 bound
are test_gpu_solver's."""
import numpy as np
import pytest

import delta2_amd as d2
from delta2_amd import scenes
from test_gpu_solver import run_case
from test_oracle_pins import record

pytestmark = pytest.mark.gpu
SHAPES = {"one": (1, 1, 1), "two floors": (1, 1, 1), "stack": (1, 1, 2), "layer": (2, 2, 1), "block": (3, 3, 2)}


def scene(counts, seed):
    rng = np.random.default_rng(seed)
    FV = np.array([[-400, -400, 0], [400, -400, 0], [400, 400, 0], [-400, 400, 0]], dtype=float)
    FF = np.array([[0, 1, 2], [0, 2, 3]], dtype=np.int32)
    V, F = scenes.icosphere(1, 0.5)
    vol, _, inertia = scenes.mass_properties(V, F)
    stream = d2.pcg_seed(42, 54)
    trees = [scenes.tree_build(FV, FF, stream), scenes.tree_build(V, F, stream)]
    ext, gap = V.max(axis=0) - V.min(axis=0), 0.003
    recs, pairs = [record(static=True, last=scenes.DT) for _ in range(2)], []
    kinds = rng.permutation(np.repeat(list(counts), list(counts.values())))
    side = int(np.ceil(np.sqrt(kinds.size)))
    for c, kind in enumerate(kinds):
        nx, ny, nz = SHAPES[kind]
        at = {}
        for z in range(nz):
            for i in range(nx):
                for j in range(ny):
                    at[i, j, z] = len(recs)
                    pos = 4.0 * np.array([c % side - side / 2, c // side - side / 2, 0]) + np.array([i, j, z]) * (ext + gap)
                    pos[2] += gap - V[:, 2].min()
                    v = (rng.normal(0, 0.03), rng.normal(0, 0.03), -0.05)
                    recs.append(record(trans=pos, vel=v, inv_inertia=np.linalg.inv(inertia), last=scenes.DT))
        for (i, j, z), b in at.items():
            if z == 0:
                pairs += [(f, b) for f in range(2 if kind == "two floors" else 1)]
            pairs += [(b, at[q]) for q in ((i + 1, j, z), (i, j + 1, z), (i, j, z + 1)) if q in at]
    pairs = np.array(pairs, dtype=np.int32)[rng.permutation(len(pairs))]
    pairs[::2] = pairs[::2, ::-1]
    rec = np.stack(recs)
    return trees, [0] * 2 + [1] * (rec.shape[0] - 2), rec, pairs, np.where(rec[:, 38] != 0, 1.0, vol)


@pytest.mark.parametrize("counts", [
    {"one": 7000, "two floors": 200, "stack": 40, "layer": 20},  # singles by lanes, the rest by blocks
    {"one": 500, "two floors": 500, "stack": 3000},              # all by lanes
    {"one": 40, "two floors": 40, "stack": 40, "layer": 20, "block": 2},  # all by blocks
])
def test_many_small_clusters(counts):
    trees, tob, rec, pairs, mass = scene(counts, sum(counts.values()))
    t = run_case(str(counts), trees, tob, rec, pairs, mass, np.full(rec.shape[0], 0.4))
    assert t["solved"] > 1.9 * sum(counts.values())
