"""FP64 products through LDS windows at the sizes from which they are taken: the
edges of tiles, wavefronts and workgroups, and a handle's two kernels on both
sides of the limit."""
import numpy as np
import pytest

from gpu_util import assert_spmv_close, to_dev
from diploma_research_amd import Csr5
from oracle import oracle as O
from test_gpu_window import _matrix

pytestmark = pytest.mark.gpu


def _lens(name, tiles, tile, rng):
    if name == "uneven, some empty":
        lens = rng.integers(1, 24, tiles * tile // 11)
        lens[rng.random(len(lens)) < 0.05] = 0
        return lens
    if name == "single elements":
        return np.ones(tiles * tile + 3, int)
    if name == "rows end with tiles":
        return np.full(tiles * tile // 8, 8)
    if name == "runs of single elements":  # tiles with more row starts than a wavefront keeps sums
        lens = np.full(tiles * tile // 15, 12)
        for at in range(500, len(lens) - 3 * tile, len(lens) // 9):
            lens[at: at + 2 * tile + 17] = 1
        return lens
    if name == "rows of three":
        return rng.integers(1, 6, tiles * tile // 3)
    if name == "rows over wavefronts":
        lens = np.full((tiles // 8 + 1) * 6, tile)
        lens[3::6] = 4 * tile
        lens[4::6] = tile // 2 + 1
        return lens
    if name == "rows over workgroups":
        return np.concatenate([rng.integers(1, 9, tiles * tile // 6), [40 * tile], rng.integers(1, 9, tiles * tile // 9)])
    raise KeyError(name)


@pytest.mark.parametrize("name", ["uneven, some empty", "single elements", "rows end with tiles",
                                  "rows over wavefronts", "rows over workgroups", "runs of single elements",
                                  "rows of three"])
@pytest.mark.parametrize("sigma,tiles", [(4, 2060), (4, 2990), (4, 6500), (7, 2060), (8, 3500), (16, 2040), (16, 2400)])
@pytest.mark.parametrize("band", [0, 6000])
def test_products_on_both_sides_of_the_limits(cuda, name, sigma, tiles, band):
    """band 0: as narrow as the rows allow."""
    rng = np.random.default_rng(sigma + tiles)
    tile = 64 * sigma
    lens = _lens(name, tiles, tile, rng)
    band = max(band, int(lens.max()))
    cols = max(len(lens) * 3 // 4, 50 * tile)
    rp, ci, v = _matrix(lens, cols, band, rng)
    rows = len(lens)
    A = Csr5.from_csr_device(rows, cols, *(to_dev(a.astype(np.int32)) for a in (rp, ci)), to_dev(v), sigma=sigma)
    x = rng.uniform(-1, 1, cols)
    used = np.zeros(cols, bool)
    used[ci] = True
    x[~used] = np.nan
    xu = np.where(used, x, 0.0)
    y = A.spmv(to_dev(x)).cpu().numpy()
    assert_spmv_close(y, O.Csr5(rows, cols, rp, ci, v).spmv(xu, nthreads=4), rp, ci, v, xu)
    assert (y[lens == 0] == 0).all()
