"""Conjugate gradients by resident workgroups: how a solve's systems are given
to teams of workgroups."""
import numpy as np
import pytest

from gpu_util import to_dev
from diploma_research_amd import Csr5, conjugate_gradient, conjugate_gradient_multi, matgen
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(40, 41), (12, 13, 14)])
@pytest.mark.parametrize("precision", ["f64", "f32-refined"])
def test_batch_of_one_system_as_a_matrix(cuda, grid, precision):
    """A batch of one system is also a matrix of its own: the single and the
    several-column solves take its system's diagonals."""
    rp, ci, v = matgen.varcoef(grid, 0.5, seed=4)
    n = len(rp) - 1
    B = np.random.default_rng(4).uniform(-1, 1, (n, 2))
    A = Csr5.from_csr_batched([(n, rp, ci, v)], sigma=8, keep_f32=True)
    M = O.Csr5(n, n, rp, ci, v)
    x, r = conjugate_gradient(A, to_dev(B[:, 0].copy()), rtol=1e-10, max_iters=2000, precision=precision)
    X, R = conjugate_gradient_multi(A, to_dev(B), rtol=1e-10, max_iters=2000, precision=precision)
    for j, (xj, rj) in enumerate([(x, r), (X[:, 1], R[1])]):
        oc = M.cg(B[:, j].copy(), rtol=1e-10, maxit=2000)
        assert rj.converged and rj.relres_true <= 1.01e-10
        np.testing.assert_allclose(xj.cpu().numpy(), oc["x"], rtol=1e-6, atol=1e-7)
