"""GPU: the broad phase with many static bodies, each sweeping the bodies after
it in several segments, at each segment length the upload chooses (512 bodies
while there are few segments, up to 4096): pair lists and clusters equal the
oracle's, as integers."""
import numpy as np
import pytest

from broad_cases import particle
from test_gpu_broad_batches import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_static,side", [
    (700, 350, 30.0),      # 512 bodies a segment, one or two each
    (6000, 4000, 70.0),    # 512, up to twelve each
    (20000, 3000, 110.0),  # 1024
    (20000, 9000, 110.0),  # 4096
    (9000, 8990, 80.0),    # nearly all static
])
def test_static_heavy(n, n_static, side):
    rng = np.random.default_rng(n_static)
    static = np.zeros(n, dtype=bool)
    static[rng.permutation(n)[:n_static]] = True
    static[0], static[-1] = True, n_static > n // 2  # a sweep over all others; one over none
    pairs = check(np.stack([particle(pos=rng.uniform(0, side, size=3), static=bool(s)) for s in static]))
    assert pairs > 5
