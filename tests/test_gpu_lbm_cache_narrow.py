"""The collide-stream's cached population planes with narrow channels: the last
batch that has all of them cached, and the first with none (their counts are
asserted in test_launch_rules.py)."""
import numpy as np
import pytest

from test_gpu_lbm_cache import advance

pytestmark = pytest.mark.gpu


def test_narrow_batches_around_the_limit():
    (want,), _ = [x[:1] for x in advance(32, 256, "fp32", 1, True)]
    for copies in (129, 130):  # 228.3 and 230.03 MB
        lbm, _ = advance(32, 256, "fp32", copies, True)
        for got in lbm:
            for a, b in zip(got, want):
                assert np.array_equal(a, b), copies
