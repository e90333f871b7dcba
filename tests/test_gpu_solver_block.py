"""GPU: the block form of the solver at the sizes where it changes hands --
clusters above the LDS capacity (192 contacts, 64 particles), levels wider than
one wavefront (more than 32 independent contacts), a cluster of more than 1024
pairs, several static bodies in one cluster, and many small clusters --
against the oracle's sequential walk, over two steps (the second warm-started).
The comparison and its 1e-9 bound are test_gpu_solver's."""
import numpy as np
import pytest

import delta2_amd as d2
from delta2_amd import scenes
from test_gpu_solver import run_case
from test_oracle_pins import record

pytestmark = pytest.mark.gpu


def floor_grid(nx, ny, layers, floors=1, gap=0.003, touch=True, seed=9):
    """nx x ny x layers spheres (subdivision 1) a gap apart over `floors`
    coplanar static floors; touch=False spreads them so that every sphere is a
    cluster of its own with the floor."""
    rng = np.random.default_rng(seed)
    FV = np.array([[-40, -40, 0], [40, -40, 0], [40, 40, 0], [-40, 40, 0]], dtype=float)
    FF = np.array([[0, 1, 2], [0, 2, 3]], dtype=np.int32)
    V, F = scenes.icosphere(1, 0.5)
    vol, _, inertia = scenes.mass_properties(V, F)
    stream = d2.pcg_seed(42, 54)
    trees = [scenes.tree_build(FV, FF, stream), scenes.tree_build(V, F, stream)]
    recs = [record(trans=(0, 0, 0), static=True, last=scenes.DT) for _ in range(floors)]
    ext = (V.max(axis=0) - V.min(axis=0) + gap) * (1.0 if touch else 1.5)
    low = -float(V[:, 2].min()) + gap
    for z in range(layers):
        for i in range(nx):
            for j in range(ny):
                pos = ((i - nx / 2) * ext[0], (j - ny / 2) * ext[1], low + z * ext[2])
                v = (rng.normal(0, 0.03), rng.normal(0, 0.03), -0.05)
                recs.append(record(trans=pos, vel=v, inv_inertia=np.linalg.inv(inertia), last=scenes.DT))
    rec = np.stack(recs)
    radii = np.concatenate([np.full(floors, 60.0), np.full(rec.shape[0] - floors, 0.5)])
    return trees, [0] * floors + [1] * (rec.shape[0] - floors), rec, scenes.broad_phase(rec, radii), np.where(
        rec[:, 38] != 0, 1.0, vol)


@pytest.mark.parametrize("nx,ny,layers,floors,least", [
    (3, 3, 2, 1, 20),      # LDS, one wavefront
    (5, 5, 2, 1, 60),      # near the LDS capacities
    (9, 9, 1, 2, 100),     # above 64 particles: global scratch, two floors
    (24, 22, 1, 1, 1000),  # above 1024 pairs and levels wider than 32
])
def test_settling_grid(nx, ny, layers, floors, least):
    trees, tob, rec, pairs, mass = floor_grid(nx, ny, layers, floors)
    if floors > 1:
        pairs = pairs[(rec[pairs, 38] == 0).any(axis=1)]
    t = run_case(f"grid {nx}x{ny}x{layers}", trees, tob, rec, pairs, mass, np.full(rec.shape[0], 0.4))
    assert t["contacts"] >= least


def test_separate_spheres():
    trees, tob, rec, pairs, mass = floor_grid(4, 4, 1, touch=False)
    pairs[::2] = pairs[::2, ::-1]  # either body first
    t = run_case("apart", trees, tob, rec, pairs, mass, np.full(rec.shape[0], 0.4))
    assert t["solved"] >= 16
