"""The launch sequences of the solvers on stencil matrices, which otherwise
iterate on resident workgroups: the workgroups are never seated here, as on a
GPU whose CUs another program holds."""
import numpy as np
import pytest

from gpu_util import to_dev
from diploma_research_amd import Csr5, conjugate_gradient, conjugate_gradient_multi, matgen
from diploma_research_amd.csr5 import conjugate_gradient_batched
from oracle import oracle as O
from test_gpu_resident_teams import NEVER_SEATED, _resident

pytestmark = pytest.mark.gpu


def _called_off(A):
    """A, whose resident launches are called off."""
    _resident(A, NEVER_SEATED)
    return A


# sides, spread of the coefficients, columns, tile height, refine_delta
@pytest.mark.parametrize("side,spread,k,sigma,delta", [(32, 1.0, 1, 16, 0.0), (32, 1.0, 4, 16, 0.0), (64, 1.0, 8, 7, 0.0),
                                                       (40, 2.0, 4, 7, 1e-30), (24, 1.0, 3, 5, 0.0)])
def test_fp32_refined(cuda, side, spread, k, sigma, delta):
    """FP32 iteration inside FP64 residual replacement, column by column
    against the oracle's FP64 CG; with a negligible refine_delta the residual is
    replaced only when FP32 says converged, and columns resume."""
    rp, ci, v = matgen.varcoef((side, side, side), spread, seed=side + k)
    n = side ** 3
    A = _called_off(Csr5.from_csr((n, n, rp, ci, v), sigma=sigma, keep_f32=True))
    B = np.random.default_rng(k).uniform(-1, 1, (n, k))
    X, res = conjugate_gradient_multi(A, to_dev(B), rtol=1e-10, max_iters=40000, precision="f32-refined",
                                      refine_delta=delta)
    assert _resident(A) == 0
    for j in range(k):
        oc = O.Csr5(n, n, rp, ci, v).cg(B[:, j].copy(), rtol=1e-10, maxit=40000, nthreads=16)
        assert res[j].converged and res[j].relres_true <= 1.01e-10
        assert res[j].iterations <= 2 * oc["iterations"] + 50
        err = np.linalg.norm(X[:, j].cpu().numpy() - oc["x"]) / np.linalg.norm(oc["x"])
        assert err < 1e-6, err
    assert res[0].refinements >= (2 if delta else 1)


def test_kept_iterations_equal_fresh_handles(cuda):
    """The captured iterations and buffers that a handle keeps, over solves of
    other vectors, columns, precisions and history lengths: the same bits as
    fresh handles."""
    import torch

    rp, ci, v = matgen.varcoef((40, 40), 0.5, seed=7)
    n = 1600
    rng = np.random.default_rng(4)
    b1, b2 = to_dev(rng.uniform(-1, 1, n)), to_dev(rng.uniform(-1, 1, n))
    B3 = to_dev(rng.uniform(-1, 1, (n, 3)))
    xbuf = torch.zeros(n, dtype=torch.float64, device="cuda")

    def make():
        return _called_off(Csr5.from_csr((n, n, rp, ci, v), sigma=5, keep_f32=True))

    def single(M, b, x=None, **kw):
        xs, r = conjugate_gradient(M, b, None if x is None else x.zero_(), rtol=1e-10, max_iters=3000, **kw)
        return xs.clone(), [r]

    steps = [
        lambda M: single(M, b1),
        lambda M: single(M, b2, xbuf),
        lambda M: single(M, b1, xbuf),  # same x buffer: the captured iterations again
        lambda M: single(M, b1, history=True),
        lambda M: single(M, b2, precision="f32-refined"),
        lambda M: conjugate_gradient_multi(M, B3, rtol=1e-10, max_iters=3000),
        lambda M: single(M, b2, xbuf, check_every=6),
        lambda M: single(M, b2, xbuf),
    ]
    A = make()
    for step in steps:
        x_kept, r_kept = step(A)
        x_new, r_new = step(make())
        assert torch.equal(x_kept, x_new)
        assert [r.iterations for r in r_kept] == [r.iterations for r in r_new]
        assert all(r.converged for r in r_kept)
    assert _resident(A) == 0


@pytest.mark.parametrize("grid,sigma", [((73, 73, 73), 7), ((87, 87, 87), 7), ((160, 160), 5), ((61, 67), 8)])
def test_coded_products_with_the_dot(cuda, grid, sigma):
    """The column-coded product with the fused p.q, in chunks of one to three
    tiles: the oracle's iteration count within 2, and the capped iterate."""
    rp, ci, v = matgen.varcoef(grid, 0.3, seed=1)
    n = len(rp) - 1
    b = np.random.default_rng(1).uniform(-1, 1, n)
    A = _called_off(Csr5.from_csr((n, n, rp, ci, v), sigma=sigma))
    assert A.info.column_codes == 1
    M = O.Csr5(n, n, rp, ci, v)
    x, r = conjugate_gradient(A, to_dev(b), rtol=1e-8, max_iters=5000)
    oc = M.cg(b, rtol=1e-8, maxit=5000, nthreads=16)
    assert r.converged and abs(r.iterations - oc["iterations"]) <= 2
    xc, rc = conjugate_gradient(A, to_dev(b), rtol=1e-14, max_iters=9)
    assert not rc.converged and rc.iterations == 9
    np.testing.assert_allclose(xc.cpu().numpy(), M.cg(b, rtol=1e-14, maxit=9, nthreads=16)["x"], rtol=1e-9, atol=1e-11)
    assert _resident(A) == 0


def test_kept_batch_iterations_equal_fresh_handles(cuda):
    """The same for a batch's captured iterations and the cooperative kernel,
    and the cap's iterate."""
    import torch

    systems = []
    for i, side in enumerate([21, 9, 33, 14]):
        rp, ci, v = matgen.varcoef((side, side), 0.5, seed=70 + i)
        systems.append((side * side, rp, ci, v))
    N = sum(n for n, *_ in systems)
    rng = np.random.default_rng(70)
    h1 = rng.uniform(-1, 1, N)
    b1, b2 = to_dev(h1), to_dev(rng.uniform(-1, 1, N))
    xbuf = torch.zeros(N, dtype=torch.float64, device="cuda")

    def make():
        return _called_off(Csr5.from_csr_batched(systems, sigma=5))

    def run(M, b, x=None, rtol=1e-11, max_iters=4000, **kw):
        X, res = conjugate_gradient_batched(M, b, None if x is None else x.zero_(), rtol=rtol, max_iters=max_iters, **kw)
        return X.clone(), res

    steps = [
        lambda M: run(M, b1),
        lambda M: run(M, b2, xbuf),
        lambda M: run(M, b1, xbuf),
        lambda M: run(M, b1, persistent=True),
        lambda M: run(M, b2, xbuf, check_every=5),
        lambda M: run(M, b1, xbuf),
        lambda M: run(M, b1, xbuf, rtol=1e-14, max_iters=17),
    ]
    A = make()
    for step in steps:
        x_kept, r_kept = step(A)
        x_new, r_new = step(make())
        assert torch.equal(x_kept, x_new)
        assert [(r.iterations, r.converged) for r in r_kept] == [(r.iterations, r.converged) for r in r_new]
    off = 0
    for (n, rp, ci, v), r in zip(systems, r_kept):
        oc = O.Csr5(n, n, rp, ci, v).cg(h1[off: off + n], rtol=1e-14, maxit=17)
        assert r.converged == oc["converged"]
        np.testing.assert_allclose(x_kept[off: off + n].cpu().numpy(), oc["x"], rtol=1e-9, atol=1e-11)
        off += n
    assert _resident(A) == 0
