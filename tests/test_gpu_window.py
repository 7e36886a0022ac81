"""Products through LDS windows: the edges of tiles, wavefronts and workgroups
(16 tiles each, or more of a large matrix), and the widths a window can have."""
import numpy as np
import pytest

from gpu_util import assert_spmv_close, to_dev
from diploma_research_amd import Csr5
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _matrix(lens, cols, band, rng):
    """Rows of the given lengths, columns within `band` of the scaled diagonal."""
    rows = len(lens)
    rp = np.zeros(rows + 1, np.uint32)
    np.cumsum(lens, out=rp[1:])
    nnz = int(rp[-1])
    row = np.repeat(np.arange(rows), lens)
    lo = np.clip(row * cols // rows - band // 2, 0, max(0, cols - band))
    k = np.arange(nnz) - rp[:-1].astype(np.int64)[row]  # element k of its row
    ci = lo + (k * band) // np.maximum(1, np.asarray(lens)[row])  # ascending, distinct while lens <= band
    return rp, ci.astype(np.uint32), rng.standard_normal(nnz)


def _lens(name, tile, rng):
    if name == "uneven, some empty":
        lens = rng.integers(1, 24, 1030 * tile // 12)
        lens[rng.random(len(lens)) < 0.05] = 0
        return lens
    if name == "single elements":  # as many row starts as a tile has places
        return np.ones(1025 * tile + 3, int)
    if name == "rows end with tiles":  # a row start at every tile's first place, the last tile full
        return np.full(1040 * tile // 4, 4)
    if name == "rows over wavefronts":  # tiles without a row start inside a workgroup
        lens = np.full(120 * 6, tile)
        lens[3::6] = 4 * tile
        lens[4::6] = tile // 2 + 1
        return lens
    if name == "rows over workgroups":  # more than a workgroup looks ahead: the tile kernel's
        return np.concatenate([rng.integers(1, 9, 700 * tile // 4), [40 * tile], rng.integers(1, 9, 400 * tile // 4)])
    if name == "many tiles":  # several tiles per wavefront
        return rng.integers(2, 9, 4200 * tile // 5)
    raise KeyError(name)


@pytest.mark.parametrize("name", ["uneven, some empty", "single elements", "rows end with tiles",
                                  "rows over wavefronts", "rows over workgroups", "many tiles"])
@pytest.mark.parametrize("sigma", [4, 7, 16])
def test_window_products(cuda, name, sigma):
    if name == "many tiles" and sigma != 4:
        sigma = 5
    rng = np.random.default_rng(sigma)
    lens = _lens(name, 64 * sigma, rng)
    cols = max(len(lens) * 3 // 4, 50 * 64 * sigma)
    rp, ci, v = _matrix(lens, cols, {"rows over wavefronts": 5, "rows over workgroups": 44}.get(name, 0) * 64 * sigma or 6000, rng)
    rows = len(lens)
    A = Csr5.from_csr_device(rows, cols, *(to_dev(a.astype(np.int32)) for a in (rp, ci)), to_dev(v), sigma=sigma,
                             keep_f32=True)
    x = rng.uniform(-1, 1, cols)
    used = np.zeros(cols, bool)
    used[ci] = True
    x[~used] = np.nan  # entries of a window that no element multiplies
    ref = O.Csr5(rows, cols, rp, ci, v).spmv(np.where(used, x, 0.0), nthreads=4)
    y = A.spmv(to_dev(x)).cpu().numpy()
    assert_spmv_close(y, ref, rp, ci, v, np.where(used, x, 0.0))
    assert (y[lens == 0] == 0).all()
    # FP32: unit roundoff 2^-24, every row a sum of products of rounded values
    y32 = A.spmv(to_dev(x.astype(np.float32))).cpu().numpy().astype(np.float64)
    rows_of = np.repeat(np.arange(rows), lens)
    absum = np.bincount(rows_of, weights=np.abs(v * np.where(used, x, 0.0)[ci]), minlength=rows)
    assert (np.abs(y32 - ref) <= (np.asarray(lens) + 4) * 2.0 ** -24 * absum + 1e-40).all()


@pytest.mark.parametrize("width", [1, 63, 12000, 16100, 16400, 32000, 40000])
def test_window_widths(cuda, width):
    """Around the widest window that FP64 (16k entries) and FP32 (36k) have room for."""
    rng = np.random.default_rng(width)
    sigma, tiles = 16, 1030
    lens = np.full(tiles * 64 * sigma // min(64, width) + 5, min(64, width))
    rows = len(lens)
    rp, ci, v = _matrix(lens, width, width, rng)
    A = Csr5.from_csr_device(rows, width, *(to_dev(a.astype(np.int32)) for a in (rp, ci)), to_dev(v), sigma=sigma,
                             keep_f32=True)
    x = rng.integers(-8, 9, width).astype(np.float64)
    w = np.rint(v * 4)
    A.set_values(to_dev(w))
    ref = O.Csr5(rows, width, rp, ci, w).spmv(x, nthreads=4)  # small whole numbers: exact in both types
    np.testing.assert_array_equal(A.spmv(to_dev(x)).cpu().numpy(), ref)
    np.testing.assert_array_equal(A.spmv(to_dev(x.astype(np.float32))).cpu().numpy(), ref.astype(np.float32))


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("name", ["uneven, some empty", "rows over workgroups", "many tiles"])
@pytest.mark.parametrize("band", [100, 6000, 20300, 20600])
def test_transposed_window_products(cuda, name, band, f32):
    """Around the widest window that a transposed product has room for (20k
    entries); columns that no window covers; whole numbers, so exact."""
    import torch

    sigma = 4 if name == "many tiles" else 16
    rng = np.random.default_rng(band)
    lens = np.minimum(_lens(name, 64 * sigma, rng), band)
    cols = band + 7000
    rp, ci, v = _matrix(lens, cols, band, rng)
    v = np.rint(v * 4)
    rows = len(lens)
    A = Csr5.from_csr_device(rows, cols, *(to_dev(a.astype(np.int32)) for a in (rp, ci)), to_dev(v), sigma=sigma,
                             keep_f32=f32)
    x = rng.integers(-8, 9, rows).astype(np.float64)
    ref = np.bincount(ci, weights=v * np.repeat(x, lens), minlength=cols)
    y = A.spmv_transpose(to_dev(x, torch.float32 if f32 else None))
    np.testing.assert_array_equal(y.cpu().numpy().astype(np.float64), ref)
    y2 = A.spmv_transpose(to_dev(-x, torch.float32 if f32 else None), torch.full_like(y, float("nan")))
    np.testing.assert_array_equal(y2.cpu().numpy().astype(np.float64), -ref)


def test_captured_window_products(cuda):
    """Both products recorded and replayed with other inputs."""
    import torch

    rng = np.random.default_rng(7)
    rp, ci, v = _matrix(_lens("uneven, some empty", 512, rng), 30000, 3000, rng)
    rows, v = len(rp) - 1, np.rint(v * 4)
    A = Csr5.from_csr_device(rows, 30000, *(to_dev(a.astype(np.int32)) for a in (rp, ci)), to_dev(v), sigma=8)
    x, u = (torch.zeros(n, dtype=torch.float64, device="cuda") for n in (30000, rows))
    y, z = torch.zeros_like(u), torch.zeros_like(x)
    A.spmv_transpose(u, z)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        A.spmv(x, y)
        A.spmv_transpose(u, z)
    row = np.repeat(np.arange(rows), np.diff(rp.astype(np.int64)))
    for _ in range(3):
        xh, uh = rng.integers(-8, 9, 30000).astype(float), rng.integers(-8, 9, rows).astype(float)
        x.copy_(to_dev(xh))
        u.copy_(to_dev(uh))
        g.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(y.cpu().numpy(), np.bincount(row, weights=v * xh[ci], minlength=rows))
        np.testing.assert_array_equal(z.cpu().numpy(), np.bincount(ci, weights=v * uh[row], minlength=30000))
