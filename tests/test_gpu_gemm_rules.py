"""The q4 large-batch GEMM on both sides of its rules: 64 weight rows a wave
(256 workgroups, or 128 with 24 groups of K) or 32, and K in one part or in
several where it has few groups, with ragged rows, columns and batches."""
import pytest

import test_gpu_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["q4t", "q4tp"])
@pytest.mark.parametrize("shape", [
    (4112, 96, 1030), (4080, 96, 1000),    # 289 and 256 workgroups of 64 rows a wave
    (2064, 3104, 1030), (2040, 2912, 1030),  # 153 with 25 groups, 136 with 23
    (1032, 1056, 449), (1000, 1056, 513),  # 32 rows a wave: 72 workgroups of 9 groups in one part, 8 more
    (1000, 1056, 500), (1000, 1440, 530),  # 64 of 9 groups in two parts, 72 of 12 groups
])
def test_gemm_rules(gpu, dt, shape):
    test_gpu_gemm.test_gemm_edges(gpu, dt, shape)
