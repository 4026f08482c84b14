"""Both sides of the rule that gives the experts' GEMVs to the kernel over
each job's own tokens or to the grouped GEMVs over all rows: q4 rows of 2048
columns by batch and jobs, of more than 3072 by tokens per expert."""
import pytest

import test_gpu_moe_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,ne,k,H,I,b", [
    ("q4tp", 64, 8, 2048, 64, 2), ("q4tp", 64, 8, 2048, 64, 3), ("q4tp", 64, 8, 2048, 64, 5), ("q4tp", 64, 8, 2048, 64, 6),
    ("q4tp", 64, 8, 1920, 64, 4), ("q4t", 40, 8, 2176, 96, 5), ("q4t", 40, 8, 2176, 96, 7),
    ("q4t", 8, 2, 3104, 64, 6), ("q4t", 8, 2, 3104, 64, 7), ("q4t", 8, 2, 3072, 64, 16), ("q4tp", 8, 2, 3104, 96, 13)])
def test_moe_rules(gpu, dt, ne, k, H, I, b):
    test_gpu_moe_rows.test_moe_rows(gpu, dt, dt, ne, k, H, I, b)
