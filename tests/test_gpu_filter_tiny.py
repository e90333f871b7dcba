"""GPU: the contact filter at search distances whose squares FP32 cannot hold
(below 1e-19) or only as subnormals: coincident contacts and contacts a search
distance apart are decided as the FP64 test decides them, in the LDS forms and
above them, against the oracle."""
import numpy as np
import pytest

import delta2_amd as d2
import d2o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("search", [0.0, 1e-300, 1e-30, 1e-24, 2e-23, 3e-22, 1e-19, 1e-15, 1e-12])
@pytest.mark.parametrize("n,spread", [(3, 0.0), (65, 0.0), (65, 1.5), (700, 0.0), (700, 1.5), (2100, 1.5)])
def test_filter_tiny_search(n, spread, search):
    """spread: the contacts lie up to that many search distances from the first."""
    rng = np.random.default_rng(n)
    r = np.zeros((n, 11))
    r[:, 0:3] = rng.uniform(-1.0, 1.0, size=(n, 3)) * spread * search
    r[:, 3:6] = r[:, 0:3]
    r[:, 6] = search
    with d2.Context(0, d2.D2_FP64) as c:
        order, kept = c.filter_contacts(r, 0.0)
    o_order, o_kept = d2o.filter_order(r, 0.0)
    assert np.array_equal(order, o_order)
    assert np.array_equal(kept, o_kept)
    if search > 1e-150:
        assert 0 < len(kept) < n  # some are dropped as near
