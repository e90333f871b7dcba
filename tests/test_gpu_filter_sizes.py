"""GPU: the contact filter at the sizes where it changes form (a wavefront's
group of 64 candidates, 256 and 1024 threads, the LDS capacities 512 and 2048,
above both) and with the inputs its shortcuts decide on -- no exact ties, many
exact ties, all keys equal -- against the oracle: whole numbers, equal."""
import numpy as np
import pytest

import delta2_amd as d2
import d2o

pytestmark = pytest.mark.gpu


def contacts(n, kind, seed):
    rng = np.random.default_rng(seed)
    r = np.zeros((n, 11))
    mid = rng.uniform(0.0, 0.4, size=(n, 3))
    half = rng.uniform(0.0, 0.01, size=n)
    eps = 0.01 + rng.uniform(0.0, 0.01, size=n)
    if kind == "ties":
        half[rng.uniform(size=n) < 0.5] = 0.0
        eps = 0.01 + rng.integers(4, size=n) * 1e-3
    if kind == "equal":
        half[:], eps[:] = 0.001, 0.015
    d = np.zeros((n, 3))
    d[:, 2] = half
    r[:, 0:3], r[:, 3:6] = mid + d, mid - d
    r[:, 6], r[:, 7] = eps, 0.01
    return r


@pytest.mark.parametrize("kind", ["apart", "ties", "equal"])
@pytest.mark.parametrize("n", [1, 2, 16, 17, 63, 64, 65, 255, 257, 512, 513, 1023, 1025, 2048, 2049, 2600])
def test_filter_sizes(n, kind):
    r = contacts(n, kind, n)
    with d2.Context(0, d2.D2_FP64) as c:
        order, kept = c.filter_contacts(r, 0.0)
    o_order, o_kept = d2o.filter_order(r, 0.0)
    assert np.array_equal(order, o_order)
    assert np.array_equal(kept, o_kept)


@pytest.mark.parametrize("case", ["far", "huge", "negative margin", "wide margin", "infinite"])
@pytest.mark.parametrize("n", [65, 700])
def test_filter_edges_of_the_distance_test(n, case):
    """Contacts exactly a search distance apart, 1 km from the origin, 1e20
    apart, and margins that leave FP32's range: the decisions stay the FP64 ones."""
    r = contacts(n, "ties", n)
    margin = {"negative margin": -0.015, "wide margin": 1e16, "infinite": float("inf")}.get(case, 0.0)
    r[1::3, 0] = r[0:-1:3, 0][: r[1::3].shape[0]] + (r[1::3, 6] + r[1::3, 7])  # a search distance away in x
    r[1::3, 3] = r[1::3, 0]
    if case == "far":
        r[:, 0:6] += np.array([1000.0, -700.0, 350.0] * 2)
    if case == "huge":
        r[::5, 0:6] *= 1e20
    with d2.Context(0, d2.D2_FP64) as c:
        order, kept = c.filter_contacts(r, margin)
    o_order, o_kept = d2o.filter_order(r, margin)
    assert np.array_equal(order, o_order)
    assert np.array_equal(kept, o_kept)
