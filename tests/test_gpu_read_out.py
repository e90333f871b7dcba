"""GPU: results reach the caller through a pinned window of two halves of 16
slots, on several threads when large: sizes below, at and above a slot, a half
and both, several reads in a row, byte for byte."""
import numpy as np
import pytest

import delta2_amd as d2
from gpu_cases import c1_scene

pytestmark = pytest.mark.gpu

REC = 40 * 8  # bytes of a body record
SLOT, HALF = 512 << 10, 8 << 20


@pytest.mark.parametrize("n", [1, 102, 103, SLOT // REC, SLOT // REC + 1, 4 * SLOT // REC + 1, HALF // REC, HALF // REC + 1,
                               2 * HALF // REC + 1, 5 * HALF // REC + 3])
def test_records_come_back(n):
    """(Other records in between: a slot is never read before it is written.)"""
    rng = np.random.default_rng(n)
    with d2.Context(0, d2.D2_FP64) as c:
        c.upload_trees(c1_scene().trees)
        for k in range(3):
            rec = rng.uniform(-1.0, 1.0, size=(n, 40))
            c.upload_bodies(np.zeros(n, dtype=np.int32), rec)
            assert np.array_equal(c.download_bodies(), rec)
