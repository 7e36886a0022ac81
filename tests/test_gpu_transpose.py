"""A^T x of matrices large enough to be sorted by column (and just below),
with integer values, for which every order of the sums is exact."""
import numpy as np
import pytest

from gpu_util import to_dev
from diploma_research_amd import Csr5, matgen

pytestmark = pytest.mark.gpu


def _exact(rp, ci, v, x, cols):
    rows = np.repeat(np.arange(len(x)), np.diff(rp.astype(np.int64)))
    return np.bincount(ci, weights=v * x[rows], minlength=cols)


# (rows, cols, longest row, share of empty rows, long rows): below and above
# the limit; one column and few columns (several workgroups to a bin); columns
# at and around a bin's 64; many bins; rows across tiles
CASES = [
    (9000, 9000, 6, 0.0, ()),
    (12000, 9000, 9, 0.1, ()),
    (70000, 1, 1, 0.2, ()),
    (40000, 63, 5, 0.0, ()),
    (40000, 65, 5, 0.3, ()),
    (20000, 20000, 12, 0.05, ((7, 15000), (19999, 9000))),
    (6000, 400000, 24, 0.0, ((0, 2000),)),
]


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("sigma", [4, 7, 16, 32])
def test_sorted_products_exact(cuda, case, sigma):
    import torch

    rows, cols, longest, empty, long_rows = CASES[case]
    rp, ci, v = matgen.random_csr(rows, cols, seed=case, max_len=min(longest, cols), empty_frac=empty,
                                  long_rows=long_rows, integer=True)
    A = Csr5.from_csr((rows, cols, rp, ci, v), sigma=sigma, keep_f32=True)
    rng = np.random.default_rng(sigma)
    for _ in range(2):
        x = rng.integers(-3, 4, rows).astype(float)
        want = _exact(rp, ci, v, x, cols)
        y = torch.full((cols,), 5.0, dtype=torch.float64, device="cuda")
        np.testing.assert_array_equal(A.spmv_transpose(to_dev(x), y).cpu().numpy(), want)
        np.testing.assert_array_equal(A.spmv_transpose(to_dev(x, torch.float32)).double().cpu().numpy(), want)
    v2 = v * 2 - 1
    A.set_values(to_dev(v2))
    np.testing.assert_array_equal(A.spmv_transpose(to_dev(x)).cpu().numpy(), _exact(rp, ci, v2, x, cols))


def test_captured_before_and_after_the_first_product(cuda):
    """A product captured before the matrix has sorted anything, and one after,
    replayed with other inputs."""
    import torch

    rows = cols = 20000
    rp, ci, v = matgen.random_csr(rows, cols, seed=3, max_len=9, integer=True)
    A = Csr5.from_csr((rows, cols, rp, ci, v), sigma=8)
    x = torch.zeros(rows, dtype=torch.float64, device="cuda")
    y = torch.zeros(cols, dtype=torch.float64, device="cuda")
    rng = np.random.default_rng(5)
    for _ in range(2):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            A.spmv_transpose(x, y)
        for _ in range(3):
            xh = rng.integers(-3, 4, rows).astype(float)
            x.copy_(to_dev(xh))
            g.replay()
            torch.cuda.synchronize()
            np.testing.assert_array_equal(y.cpu().numpy(), _exact(rp, ci, v, xh, cols))
            np.testing.assert_array_equal(A.spmv_transpose(x).cpu().numpy(), y.cpu().numpy())


def test_batches_large_enough_to_be_sorted(cuda):
    systems = []
    for s in (90, 41, 70):
        rp, ci, v = matgen.poisson2d(s)
        systems.append((s * s, rp, ci, v * np.random.default_rng(s).integers(1, 5, len(v))))
    A = Csr5.from_csr_batched(systems, sigma=8)
    x = np.random.default_rng(1).integers(-3, 4, sum(n for n, *_ in systems)).astype(float)
    y = A.spmv_transpose(to_dev(x)).cpu().numpy()
    off = 0
    for n, rp, ci, v in systems:
        np.testing.assert_array_equal(y[off: off + n], _exact(rp, ci, v, x[off: off + n], n))
        off += n
