"""Conversion on the GPU of matrices with empty rows and one to many steps of
the scan of their tiles' segment counts, against the host builder."""
import numpy as np
import pytest

from gpu_util import to_dev
from diploma_research_amd import Csr5

pytestmark = pytest.mark.gpu


# tiles of sigma 4 (256 elements): around one step's 1024 entries, and several
@pytest.mark.parametrize("tiles", [1, 1023, 1024, 1025, 20001])
def test_segment_offsets_of_many_tiles(cuda, tiles):
    rng = np.random.default_rng(tiles)
    rows, cols = max(50, tiles * 40), 1000
    lens = np.zeros(rows, int)
    full = rng.random(rows) < 0.8
    lens[full] = 8
    over = int(lens.sum()) - tiles * 256  # the last tile full, or short by less than a row
    short = np.nonzero(lens)[0]
    if over > 0:
        lens[short[: -(-over // 8)]] = 0
    else:
        lens[short[0]] += min(-over, cols // 2)
    rp = np.zeros(rows + 1, np.int64)
    np.cumsum(lens, out=rp[1:])
    row = np.repeat(np.arange(rows), lens)
    k = np.arange(rp[-1]) - rp[row]
    ci = ((row * 7 + k) % cols).astype(np.int64)
    ci = np.sort(row * cols + ci) - row * cols  # ascending within a row
    v = rng.standard_normal(len(ci))
    H = Csr5.from_csr((rows, cols, rp.astype(np.uint32), ci.astype(np.uint32), v), sigma=4)
    D = Csr5.from_csr_device(rows, cols, to_dev(rp.astype(np.int32)), to_dev(ci.astype(np.int32)), to_dev(v), sigma=4)
    fh, fd = H.format_arrays(), D.format_arrays()
    for key in fh:
        np.testing.assert_array_equal(fd[key], fh[key], err_msg=key)
    assert D.info.n_dirty_tiles == H.info.n_dirty_tiles and D.info.n_empty_rows == H.info.n_empty_rows
    x = rng.integers(-4, 5, cols).astype(float)
    w = rng.integers(-8, 9, len(ci)).astype(float)
    D.set_values(to_dev(w))
    np.testing.assert_array_equal(D.spmv(to_dev(x)).cpu().numpy(), np.bincount(row, weights=w * x[ci], minlength=rows))
