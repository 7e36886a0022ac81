"""Conversion on the GPU where a tile's walk over row_ptr can go wrong, against
the host builder's format."""
import numpy as np
import pytest

from gpu_util import to_dev
from diploma_research_amd import Csr5

pytestmark = pytest.mark.gpu


def _lens(name, rng):
    if name == "no rows hold anything":
        return np.zeros(300, int)
    if name == "one element":
        return np.array([0, 0, 1, 0])
    if name == "exact tiles":  # the last tile is full for sigma 4, 16 and 32
        return np.full(4096, 8)
    if name == "empty runs":  # runs of empty rows longer than a wavefront, at both ends, inside and between tiles
        parts = [np.zeros(200, int)]
        for i in range(40):
            parts += [rng.integers(1, 9, 30 + i), np.zeros(int(rng.integers(1, 300)), int)]
        return np.concatenate(parts + [np.zeros(5000, int)])
    if name == "one row":
        return np.array([5000])
    if name == "rows over tiles":
        return np.array([0, 3000, 0, 0, 1, 2048, 0, 4096, 7, 0])
    if name == "single elements":
        return np.ones(70000, int)
    raise KeyError(name)


@pytest.mark.parametrize("name", ["no rows hold anything", "one element", "exact tiles", "empty runs", "one row",
                                  "rows over tiles", "single elements"])
@pytest.mark.parametrize("sigma", [4, 7, 16, 32])
def test_format_equals_the_host_builders(cuda, name, sigma):
    import torch

    rng = np.random.default_rng(sigma)
    lens = _lens(name, rng)
    rows, cols = len(lens), 6000
    rp = np.zeros(rows + 1, np.uint32)
    np.cumsum(lens, out=rp[1:])
    ci = np.concatenate([np.sort(rng.choice(cols, int(n), replace=False)) for n in lens if n]
                        or [np.zeros(0, int)]).astype(np.uint32)
    v = rng.standard_normal(len(ci))
    H = Csr5.from_csr((rows, cols, rp, ci, v), sigma=sigma, keep_f32=True)
    D = Csr5.from_csr_device(rows, cols, to_dev(rp.astype(np.int32)), to_dev(ci.astype(np.int32)), to_dev(v),
                             sigma=sigma, keep_f32=True)
    fh, fd = H.format_arrays(), D.format_arrays()
    for key in fh:
        np.testing.assert_array_equal(fd[key], fh[key], err_msg=key)
    assert D.info.n_dirty_tiles == H.info.n_dirty_tiles and D.info.n_empty_rows == H.info.n_empty_rows
    x = to_dev(rng.uniform(-1, 1, cols))
    assert torch.equal(D.spmv(x), H.spmv(x))
    assert torch.equal(D.spmv(x.float()), H.spmv(x.float()))
    u, w = to_dev(rng.uniform(-1, 1, rows)), x
    assert torch.equal(D.sampled_outer(u, w), H.sampled_outer(u, w))


def test_matrices_in_the_memory_of_freed_ones(cuda):
    """Matrices of 20 to 60 MB made and freed one after another (the memory of
    the last one freed is used again), with others alive and from several
    threads: every product exact."""
    import threading

    def make(rows, seed):
        rng = np.random.default_rng(seed)
        rp = (np.arange(rows + 1) * 8).astype(np.int32)
        ci = rng.integers(0, rows, rows * 8).astype(np.int32)
        v = rng.integers(-8, 9, rows * 8).astype(float)
        x = rng.integers(-4, 5, rows).astype(float)
        return rp, ci, v, x, (v * x[ci]).reshape(rows, 8).sum(1)

    def check(cases, on_gpu):
        for rp, ci, v, x, want in cases:
            rows = len(rp) - 1
            if on_gpu:
                A = Csr5.from_csr_device(rows, rows, to_dev(rp), to_dev(ci), to_dev(v), sigma=16)
            else:
                A = Csr5.from_csr((rows, rows, rp, ci, v), sigma=8)
            for _ in range(2):
                np.testing.assert_array_equal(A.spmv(to_dev(x)).cpu().numpy(), want)
            del A

    cases = [make(rows, i) for i, rows in enumerate([200_000, 210_000, 190_000, 500_000, 480_000, 200_003])]
    alive = Csr5.from_csr_device(200_000, 200_000, *(to_dev(a) for a in cases[0][:3]), sigma=16)
    check(cases, True)
    check(cases[::-1], False)
    failed = []

    def worker(part):
        try:
            for _ in range(3):
                check(part, True)
        except Exception as e:  # noqa: BLE001
            failed.append(e)

    threads = [threading.Thread(target=worker, args=(cases[i::3],)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed[0]
    np.testing.assert_array_equal(alive.spmv(to_dev(cases[0][3])).cpu().numpy(), cases[0][4])
