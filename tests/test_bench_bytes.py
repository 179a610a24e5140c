"""bench.py's algorithmic plane bytes follow the layouts the library prepares."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))


@pytest.mark.parametrize("m", [1, 2, 3, 4, 8])
@pytest.mark.parametrize("q8", [True, False])
def test_plane_bytes_match_the_prepared_planes(gh, m, q8):
    import bench

    k, n = 4096, 128
    weights, outputs = n * k // 2 + n * k // 16, m * n * 4
    planes = gh.lib().glacier_hip_activation_bytes(m, k, gh.ACT_Q8 if q8 else gh.ACT_F32)
    assert bench.gemv_bytes(n, k, m, q8) == weights + planes + outputs
