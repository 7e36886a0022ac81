"""Products of matrices kept by diagonals, against the tile kernels' bits and
the oracle."""
import numpy as np
import pytest

from gpu_util import assert_spmv_close, to_dev
from diploma_research_amd import Csr5
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _diagonals(rows, cols, offs, seed, drop=0.0, integer=False):
    """CSR of the full diagonals `offs`, less a share `drop` of the elements
    (every row keeps one)."""
    rng = np.random.default_rng(seed)
    i = np.repeat(np.arange(rows), len(offs))
    j = i + np.tile(np.asarray(offs), rows)
    ok = (j >= 0) & (j < cols)
    gone = ok & (rng.random(len(j)) < drop)
    held = np.bincount(i[ok & ~gone], minlength=rows)
    gone &= held[i] > 0
    i, j = i[ok & ~gone], j[ok & ~gone]
    rp = np.zeros(rows + 1, np.uint32)
    np.cumsum(np.bincount(i, minlength=rows), out=rp[1:])
    v = rng.integers(-8, 9, len(j)).astype(float) if integer else rng.standard_normal(len(j))
    return rp, j.astype(np.uint32), v


# (rows, cols, offsets): one to nine diagonals (kernels of 3, 5, 7 and 9),
# rows at and around the blocks of 256, rectangular both ways
CASES = [
    (1, 1, [0]),
    (255, 255, [-1, 0, 1]),
    (256, 256, [-16, -1, 0, 1, 16]),
    (257, 400, [0, 1, 17, 143]),
    (1000, 990, [-100, -10, -1, 0, 1, 10]),
    (4097, 4097, [-256, -16, -1, 0, 1, 16, 256]),
    (20011, 20011, [-142, -141, -140, -1, 0, 1, 140, 141, 142]),
]


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("drop", [0.0, 0.1])
@pytest.mark.parametrize("sigma", [7, 8, 16])
def test_products_equal_the_tile_kernels(cuda, case, drop, sigma):
    """The diagonal form sums each row in the tile kernels' order: y has the
    same bits as the plain format's, FP64 and FP32, before and after new
    values. Products of several columns against the oracle."""
    import torch

    rows, cols, offs = CASES[case]
    rp, ci, v = _diagonals(rows, cols, offs, seed=case, drop=drop)
    A = Csr5.from_csr((rows, cols, rp, ci, v), sigma=sigma, keep_f32=True)
    B = Csr5.from_csr((rows, cols, rp, ci, v), sigma=sigma, keep_f32=True, plain_columns=True)
    rng = np.random.default_rng(case + 50)
    x = rng.uniform(-1, 1, cols)
    for vals in (v, rng.standard_normal(len(v))):
        A.set_values(to_dev(vals))
        B.set_values(to_dev(vals))
        for dt in (torch.float64, torch.float32):
            assert torch.equal(A.spmv(to_dev(x, dt)), B.spmv(to_dev(x, dt)))
        for k in (2, 3, 5, 8, 16):
            X = rng.uniform(-1, 1, (cols, k))
            for Xd in (to_dev(X), to_dev(X).t().contiguous().t()):
                Y = A.spmm(Xd).cpu().numpy()
                for j in range(k):
                    assert_spmv_close(Y[:, j], O.csr_spmv(rp, ci, vals, X[:, j].copy()), rp, ci, vals, X[:, j])


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 7, 11, 16])
@pytest.mark.parametrize("f32", [False, True])
def test_columns_exact_at_any_alignment(cuda, k, f32):
    """Integer inputs are exact: row-major blocks that begin at an odd element
    of their storage, and column-major ones with a longer leading dimension."""
    import torch

    n = 2023
    rp, ci, v = _diagonals(n, n, [-45, -1, 0, 1, 45], seed=k, integer=True)
    A = Csr5.from_csr((n, n, rp, ci, v), sigma=8, keep_f32=True)
    X = np.random.default_rng(k).integers(-4, 5, (n, k)).astype(float)
    want = np.stack([O.csr_spmv(rp, ci, v, X[:, j].copy()) for j in range(k)], 1)
    dt = torch.float32 if f32 else torch.float64
    buf = torch.zeros(n * k + 1, dtype=dt, device="cuda")
    out = torch.full((n * k + 2,), 77.0, dtype=dt, device="cuda")
    Xr, Yr = buf[1:].view(n, k), out[1:-1].view(n, k)
    Xr.copy_(to_dev(X, dt))
    A.spmm(Xr, Yr)
    np.testing.assert_array_equal(Yr.double().cpu().numpy(), want)
    assert float(out[0]) == 77.0 and float(out[-1]) == 77.0
    Xc = torch.zeros((k, n + 3), dtype=dt, device="cuda")
    Xc[:, :n] = to_dev(X, dt).t()
    np.testing.assert_array_equal(A.spmm(Xc[:, :n].t()).double().cpu().numpy(), want)


def test_missing_elements_do_not_read_x(cuda):
    """NaN and infinity in x reach only the rows that hold an element there."""
    import torch

    n = 1500
    rp, ci, v = _diagonals(n, n, [-30, -1, 0, 1, 30], seed=3, drop=0.1)
    A = Csr5.from_csr((n, n, rp, ci, v), sigma=8)
    x = np.random.default_rng(4).uniform(-1, 1, n)
    x[[0, 77, 700, n - 1]] = [np.inf, np.nan, -np.inf, np.nan]
    rows = np.repeat(np.arange(n), np.diff(rp.astype(np.int64)))
    hit = np.unique(rows[np.isin(ci, [0, 77, 700, n - 1])])
    for y in (A.spmv(to_dev(x)), A.spmm(torch.stack([to_dev(x)] * 3, 1))[:, 2]):
        np.testing.assert_array_equal(np.nonzero(~np.isfinite(y.cpu().numpy()))[0], hit)


def test_unordered_columns_keep_the_tile_kernels(cuda):
    """Rows whose columns descend, or hold one column twice, are not kept by
    diagonals: their products follow the stored order."""
    n = 600
    rp, ci, v = _diagonals(n, n, [-1, 0, 1], seed=5, integer=True)
    x = np.random.default_rng(6).integers(-4, 5, n).astype(float)
    swapped = ci.copy()
    swapped[rp[40]: rp[41]] = swapped[rp[40]: rp[41]][::-1]
    twice = ci.copy()
    twice[rp[50] + 1] = twice[rp[50]]
    for cols in (swapped, twice):
        A = Csr5.from_csr((n, n, rp, cols, v), sigma=8)
        np.testing.assert_array_equal(A.spmv(to_dev(x)).cpu().numpy(), O.csr_spmv(rp, cols, v, x))
