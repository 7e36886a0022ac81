"""What bench.py says of the headline's kernel, without a GPU."""
import json
import os

import pytest

import bench


@pytest.mark.parametrize("sigma", [4, 5, 6, 7, 8, 16])
def test_kernel_of_the_headline(sigma):
    """The diagonal form takes the 7-point operator's products where its 7
    diagonals are no more than sigma; at sigma 6 the coded tile kernel runs."""
    assert bench.by_diagonals(sigma) == (7 <= sigma)
    assert not bench.by_diagonals(sigma, plain_columns=True)
    with open(os.path.join(bench.ROOT, "profiles", "spmv_tiles_f64_poisson128_traffic.json")) as f:
        by_kernel = json.load(f)["by_kernel"]
    codes = sigma <= 8
    key = "dia" if sigma >= 7 else f"{sigma}c"
    assert bench.traffic_for(sigma, codes) == by_kernel[key]["hbm_bytes_per_launch"]
    assert bench.traffic_for(sigma, False, plain_columns=True) == by_kernel[str(sigma)]["hbm_bytes_per_launch"]
