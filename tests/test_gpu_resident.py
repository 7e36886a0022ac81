"""Conjugate gradients by resident workgroups (matrices kept by diagonals)
against the oracle's CG, at the sizes where the rows are shared out
differently."""
import numpy as np
import pytest

from gpu_util import to_dev
from diploma_research_amd import Csr5, DimError, conjugate_gradient, conjugate_gradient_multi, matgen
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# grid: one wavefront; less and more than one workgroup's 1024 rows; a team
# whose last workgroup is short; 32 workgroups of an XCD with the far planes
# outside the halo; the most rows an XCD takes and one more (the whole chip);
# the whole chip with far planes and values read in every iteration
GRIDS = [(7, 9), (31, 33), (33, 32), (61, 67), (32, 32, 33), (45, 46, 47), (362, 362), (363, 362), (64, 65, 63),
         (103, 104, 105)]


def _problem(grid, seed):
    rp, ci, v = matgen.varcoef(grid, 0.5, seed=seed)
    n = len(rp) - 1
    x = np.random.default_rng(seed).uniform(-1, 1, n)
    return n, rp, ci, v, O.csr_spmv(rp, ci, v, x)


@pytest.mark.parametrize("grid", GRIDS)
def test_solution_and_capped_iterates(cuda, grid):
    """The oracle's solution at the same stop test; after 9 iterations, the
    oracle's iterate; twice the same bits."""
    import torch

    n, rp, ci, v, b = _problem(grid, seed=len(grid) * 100 + grid[0])
    A = Csr5.from_csr((n, n, rp, ci, v), sigma=8)
    M = O.Csr5(n, n, rp, ci, v)
    x, r = conjugate_gradient(A, to_dev(b), rtol=1e-10, max_iters=5000)
    oc = M.cg(b, rtol=1e-10, maxit=5000, nthreads=8)
    assert r.converged and oc["converged"]
    assert r.relres_true <= 1.01e-10
    np.testing.assert_allclose(x.cpu().numpy(), oc["x"], rtol=1e-7, atol=1e-8)
    x2, _ = conjugate_gradient(A, to_dev(b), rtol=1e-10, max_iters=5000)
    assert torch.equal(x, x2)
    xc, rc = conjugate_gradient(A, to_dev(b), rtol=1e-14, max_iters=9)
    oc = M.cg(b, rtol=1e-14, maxit=9, nthreads=8)
    assert not rc.converged and rc.iterations == 9
    np.testing.assert_allclose(xc.cpu().numpy(), oc["x"], rtol=1e-9, atol=1e-11)


@pytest.mark.parametrize("grid,k", [((40, 41), 3), ((32, 32, 33), 9), ((64, 64, 33), 8), ((364, 363), 2)])
@pytest.mark.parametrize("precision", ["f64", "f32-refined"])
def test_columns_stop_one_by_one(cuda, grid, k, precision):
    """Several right-hand sides (more than the XCDs, and larger than an XCD's
    share): every column as its own solve, at its own iteration count."""
    n, rp, ci, v, _ = _problem(grid, seed=k)
    A = Csr5.from_csr((n, n, rp, ci, v), sigma=8, keep_f32=True)
    B = np.random.default_rng(k).uniform(-1, 1, (n, k))
    B[:, 1] = 0.0  # converged at the start
    X, res = conjugate_gradient_multi(A, to_dev(B), rtol=1e-10, max_iters=5000, precision=precision)
    X = X.cpu().numpy()
    assert res[1].iterations == 0 and not X[:, 1].any()
    for j in {0, (k // 2 + 1) % k, k - 1} - {1}:
        oc = O.Csr5(n, n, rp, ci, v).cg(B[:, j].copy(), rtol=1e-10, maxit=5000, nthreads=8)
        assert res[j].converged and res[j].relres_true <= 1.01e-10
        np.testing.assert_allclose(X[:, j], oc["x"], rtol=1e-6, atol=1e-7)


@pytest.mark.parametrize("precision", ["f64", "f32-refined"])
def test_indefinite_matrix_breaks_down(cuda, precision):
    n, rp, ci, v, b = _problem((50, 50), seed=3)
    A = Csr5.from_csr((n, n, rp, ci, -v), sigma=8, keep_f32=True)
    with pytest.raises(DimError, match="breakdown"):
        conjugate_gradient(A, to_dev(b), precision=precision)


@pytest.mark.parametrize("sides", [[9] * 7 + [33], [5, 8, 40, 13] * 75, [350, 300, 20, 3, 280, 64, 64, 90, 340, 12]],
                         ids=["eight", "take turns", "uneven"])
def test_batches(cuda, sides):
    """A batch of a system per XCD, of more systems than an XCD has
    workgroups, and of very uneven ones: every system's solution, the capped
    iterate, and the persistent form's bits."""
    import torch

    from diploma_research_amd.csr5 import conjugate_gradient_batched

    systems = []
    for i, s in enumerate(sides):
        rp, ci, v = matgen.varcoef((max(3, s * 3 // 4), s), 0.5, seed=i)
        systems.append((len(rp) - 1, rp, ci, v))
    A = Csr5.from_csr_batched(systems, sigma=5)
    rng = np.random.default_rng(len(sides))
    bs = [rng.uniform(-1, 1, n) for n, *_ in systems]
    b = to_dev(np.concatenate(bs))
    X, res = conjugate_gradient_batched(A, b, rtol=1e-10, max_iters=5000)
    Xp, resp = conjugate_gradient_batched(A, b, rtol=1e-10, max_iters=5000, persistent=True)
    assert torch.equal(X, Xp) and [r.iterations for r in res] == [r.iterations for r in resp]
    Xc, resc = conjugate_gradient_batched(A, b, rtol=1e-14, max_iters=6)
    X, Xc = X.cpu().numpy(), Xc.cpu().numpy()
    off = 0
    for i, ((n, rp, ci, v), bb) in enumerate(zip(systems, bs)):
        if i < 12:
            M = O.Csr5(n, n, rp, ci, v)
            oc = M.cg(bb, rtol=1e-10, maxit=5000, nthreads=8)
            assert res[i].converged and res[i].relres_true <= 1.01e-10
            np.testing.assert_allclose(X[off: off + n], oc["x"], rtol=1e-7, atol=1e-8)
            oc = M.cg(bb, rtol=1e-14, maxit=6, nthreads=8)
            assert not resc[i].converged and resc[i].iterations == 6
            np.testing.assert_allclose(Xc[off: off + n], oc["x"], rtol=1e-9, atol=1e-11)
        off += n
