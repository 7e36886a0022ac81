"""Device memory that outlives a matrix."""
import numpy as np
import pytest

from gpu_util import to_dev
from diploma_research_amd import Csr5, release_memory

pytestmark = pytest.mark.gpu


def test_kept_block_is_given_back(cuda):
    """The arrays of a destroyed matrix stay for the next one; release_memory()
    gives them back, and matrices made after it are whole."""
    import torch

    rows = 500_000
    rng = np.random.default_rng(0)
    rp = (np.arange(rows + 1) * 8).astype(np.int32)
    ci = rng.integers(0, rows, rows * 8).astype(np.int32)
    v = rng.integers(-8, 9, rows * 8).astype(float)
    x = rng.integers(-4, 5, rows).astype(float)
    want = (v * x[ci]).reshape(rows, 8).sum(1)
    d, xd = [to_dev(a) for a in (rp, ci, v)], to_dev(x)

    def free():
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0]

    def product():
        A = Csr5.from_csr_device(rows, rows, *d, sigma=16)
        np.testing.assert_array_equal(A.spmv(xd).cpu().numpy(), want)

    product()  # (whatever a first product loads and allocates for good)
    release_memory()
    before = free()
    product()
    kept = before - free()
    assert kept >= 16 << 20  # 12 bytes per element of 4M
    release_memory()
    assert before - free() <= 4 << 20
    release_memory()  # nothing is kept: nothing happens
    product()
    product()
    release_memory()
    assert before - free() <= 4 << 20
