"""New values of matrices kept by diagonals: products, solves and batches are
those of a matrix built with them."""
import numpy as np
import pytest

from gpu_util import to_dev
from diploma_research_amd import Csr5, conjugate_gradient, matgen
from diploma_research_amd.csr5 import conjugate_gradient_batched

pytestmark = pytest.mark.gpu

# diagonals (the fifth form is not symmetric: its solves do not converge, but
# alike); the share of the places off the main one that is missing
FORMS = [([-1, 0, 1], 0.0), ([-40, -1, 0, 1, 40], 0.0), ([-40, -1, 0, 1, 40], 0.1), ([-900, -30, -1, 0, 1, 30, 900], 0.0),
         ([-900, -30, -2, -1, 0, 1, 30, 900], 0.03), ([-31, -30, -29, -1, 0, 1, 29, 30, 31], 0.0)]


def _banded(n, offs, drop, rng):
    """Values of a symmetric matrix (where the diagonals are), positive definite
    by its main diagonal."""
    at = np.arange(n)[:, None] + np.asarray(offs)[None, :]
    held = (at >= 0) & (at < n)
    up = {o: rng.uniform(0.1, 1.0, n) * (rng.random(n) >= drop) for o in offs if o > 0}
    v = np.empty(at.shape)
    for j, o in enumerate(offs):
        if o > 0:
            v[:, j] = -up[o]
        elif o < 0:
            v[:, j] = -np.roll(up.get(-o, np.ones(n)), -o)
    j0 = offs.index(0)
    v[:, j0] = 0.0
    v[~held] = 0.0
    held &= (v != 0.0) | (np.asarray(offs) == 0)
    v[:, j0] = 1.0 + np.abs(v).sum(1)
    rp = np.concatenate([[0], np.cumsum(held.sum(1))]).astype(np.uint32)
    return rp, at[held].astype(np.uint32), v[held]


@pytest.mark.parametrize("form", range(len(FORMS)))
@pytest.mark.parametrize("sigma", [4, 5, 7, 8, 16, 32])
@pytest.mark.parametrize("n", [1000, 1500, 20011])
def test_new_values_of_a_matrix(cuda, form, sigma, n):
    import torch

    offs, drop = FORMS[form]
    rng = np.random.default_rng(form * 100 + sigma)
    rp, ci, v = _banded(n, offs, drop, rng)
    A = Csr5.from_csr((n, n, rp, ci, np.full(len(ci), np.nan)), sigma=sigma, keep_f32=True)
    B = Csr5.from_csr((n, n, rp, ci, v), sigma=sigma, keep_f32=True)
    A.set_values(to_dev(v))
    x = to_dev(rng.uniform(-1, 1, n))
    assert torch.equal(A.spmv(x), B.spmv(x))
    assert torch.equal(A.spmv(x.float()), B.spmv(x.float()))
    for precision in ("f64", "f32-refined"):
        xa, ra = conjugate_gradient(A, x, rtol=1e-10, precision=precision)
        xb, rb = conjugate_gradient(B, x, rtol=1e-10, precision=precision)
        assert ra.converged or form == 4
        assert ra.iterations == rb.iterations and torch.equal(xa, xb)


@pytest.mark.parametrize("sigma", [5, 16])
def test_new_values_of_a_batch(cuda, sigma):
    """Systems with different numbers of diagonals and ragged ends."""
    import torch

    rng = np.random.default_rng(sigma)
    systems = []
    for n, (offs, drop) in zip([1, 700, 1500, 64, 257, 3001], [FORMS[0]] + FORMS[:5]):
        systems.append((n, *_banded(n, offs, drop, rng)))
    for i, side in enumerate([3, 40, 77]):
        rp, ci, v = matgen.varcoef((side, side + 1), 0.5, seed=i)
        systems.append((len(rp) - 1, rp, ci, v))
    A = Csr5.from_csr_batched([(n, rp, ci, np.full(len(ci), np.nan)) for n, rp, ci, _ in systems], sigma=sigma)
    B = Csr5.from_csr_batched(systems, sigma=sigma)
    A.set_values(to_dev(np.concatenate([v for *_, v in systems])))
    b = to_dev(rng.uniform(-1, 1, sum(n for n, *_ in systems)))
    xa, ra = conjugate_gradient_batched(A, b, rtol=1e-10)
    xb, rb = conjugate_gradient_batched(B, b, rtol=1e-10)
    assert all(r.converged for i, r in enumerate(ra) if i != 5)
    assert [r.iterations for r in ra] == [r.iterations for r in rb] and torch.equal(xa, xb)
