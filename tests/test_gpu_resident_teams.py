"""Conjugate gradients by resident workgroups: how a solve's systems are given
to teams of workgroups."""
import numpy as np
import pytest

from gpu_util import to_dev
from diploma_research_amd import Csr5, DimError, conjugate_gradient, conjugate_gradient_multi, matgen
from diploma_research_amd import native as N
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


# Three diagonals, FP64: a workgroup takes up to 8192 rows, and its window has
# room for a halo of 1408 entries.
@pytest.mark.parametrize("rows,off", [(6000, 1500), (8192, 1408), (8192, 1409), (8128, 1600)])
def test_far_diagonals_of_one_workgroup(cuda, rows, off):
    """So many systems that most teams are one workgroup, with diagonals that
    reach past its window but not past its rows: every system's solution."""
    from diploma_research_amd.csr5 import conjugate_gradient_batched

    S = 200
    rng = np.random.default_rng(rows + off)
    r = np.arange(rows)
    at = np.stack([r - off, r, r + off], 1)
    held = (at >= 0) & (at < rows)
    rp = np.concatenate([[0], np.cumsum(held.sum(1))]).astype(np.uint32)
    ci = at[held].astype(np.uint32)
    systems, xs, bs = [], [], []
    for _ in range(S):
        # symmetric: the coupling of rows i and i + off is w[i]; diagonally dominant
        w = rng.uniform(0.5, 1.0, rows)
        vals = np.stack([-np.roll(w, off), np.full(rows, 2.5), -w], 1)
        v = vals[held]
        x = rng.uniform(-1, 1, rows)
        systems.append((rows, rp, ci, v))
        xs.append(x)
        bs.append(O.csr_spmv(rp, ci, v, x))
    A = Csr5.from_csr_batched(systems, sigma=5)
    X, res = conjugate_gradient_batched(A, to_dev(np.concatenate(bs)), rtol=1e-12, max_iters=300)
    assert all(q.converged and q.relres_true <= 1.01e-12 for q in res)
    # ||A^-1|| <= 2 and ||A|| <= 4.5: the error is at most 9 times the residual's share
    x = np.concatenate(xs)
    assert np.linalg.norm(X.cpu().numpy() - x) <= 1e-11 * np.linalg.norm(x)


# The faults that the tests' hold on a handle can set
NONE, NEVER_SEATED, WAITS_FAIL = range(3)


def _resident(A, fault=NONE, start=0):
    """Resident launches of A's solves that iterated since the last call;
    those from the next but `start` on fail."""
    return N.lib().dim_test_resident(A._h, fault, start)


# one team on an XCD; the whole chip
@pytest.mark.parametrize("grid", [(61, 67), (103, 104, 105)])
def test_failed_wait_stops_every_workgroup(cuda, grid):
    """One workgroup stays away from the meetings: the waits for it end by their
    limit and stop every workgroup, the solve reports it, x keeps what it held,
    and the next solve is as ever."""
    import torch

    rp, ci, v = matgen.varcoef(grid, 0.5, seed=9)
    n = len(rp) - 1
    b = to_dev(np.random.default_rng(9).uniform(-1, 1, n))
    A = Csr5.from_csr((n, n, rp, ci, v), sigma=8)
    x0 = torch.linspace(-1, 1, n, dtype=torch.float64, device="cuda")
    _resident(A, WAITS_FAIL)
    x = x0.clone()
    with pytest.raises(DimError, match="timed out"):
        conjugate_gradient(A, b, x=x, rtol=1e-10, max_iters=3000)
    assert torch.equal(x, x0)
    assert _resident(A) == 0
    x, r = conjugate_gradient(A, b, x=x, rtol=1e-10, max_iters=3000)
    assert _resident(A) == 1
    assert r.converged and r.relres_true <= 1.01e-10


@pytest.mark.parametrize("precision", ["f64", "f32-refined"])
def test_never_seated_takes_the_launch_sequence(cuda, precision):
    """Workgroups that are not all running call the launch off: the launch
    sequence solves, single systems and batches alike."""
    from diploma_research_amd.csr5 import conjugate_gradient_batched

    rp, ci, v = matgen.varcoef((40, 41), 0.5, seed=2)
    n = len(rp) - 1
    b = np.random.default_rng(2).uniform(-1, 1, n)
    oc = O.Csr5(n, n, rp, ci, v).cg(b, rtol=1e-10, maxit=2000)
    A = Csr5.from_csr((n, n, rp, ci, v), sigma=8, keep_f32=True)
    _resident(A, NEVER_SEATED)
    x, r = conjugate_gradient(A, to_dev(b), rtol=1e-10, max_iters=2000, precision=precision)
    assert _resident(A) == 0
    assert r.converged and r.relres_true <= 1.01e-10
    np.testing.assert_allclose(x.cpu().numpy(), oc["x"], rtol=1e-6, atol=1e-7)
    if precision == "f64":
        S = Csr5.from_csr_batched([(n, rp, ci, v)] * 3, sigma=8)
        _resident(S, NEVER_SEATED)
        X, R = conjugate_gradient_batched(S, to_dev(np.tile(b, 3)), rtol=1e-10, max_iters=2000)
        assert _resident(S) == 0
        assert all(q.converged for q in R)
        np.testing.assert_allclose(X.cpu().numpy(), np.tile(oc["x"], 3), rtol=1e-7, atol=1e-8)


@pytest.mark.parametrize("k", [1, 3])
def test_called_off_after_a_refinement(cuda, k):
    """The launch sequence takes over where the resident launches end in the
    middle of an FP32-refined solve: the columns' counts, the history and the
    cap are those of one solve."""
    rp, ci, v = matgen.varcoef((40, 41), 0.5, seed=6)
    n = len(rp) - 1
    B = np.random.default_rng(6).uniform(-1, 1, (n, k)) * 10.0 ** -np.arange(k)
    A = Csr5.from_csr((n, n, rp, ci, v), sigma=8, keep_f32=True)

    def run(max_iters, **kw):
        if k == 1:
            x, r = conjugate_gradient(A, to_dev(B[:, 0].copy()), rtol=1e-10, max_iters=max_iters, **kw)
            return x[:, None], [r]
        return conjugate_gradient_multi(A, to_dev(B), rtol=1e-10, max_iters=max_iters, **kw)

    hist = {"history": True} if k == 1 else {}
    X0, R0 = run(2000, precision="f32-refined", **hist)
    assert _resident(A, NEVER_SEATED, 1) > 1
    X1, R1 = run(2000, precision="f32-refined", **hist)
    assert _resident(A, NEVER_SEATED, 1) == 1
    for j in range(k):
        assert R1[j].converged and R1[j].relres_true <= 1.01e-10
        # the forms round differently, which moves a stop by a few steps
        assert abs(R1[j].iterations - R0[j].iterations) <= 0.03 * R0[j].iterations + 3
        oc = O.Csr5(n, n, rp, ci, v).cg(B[:, j].copy(), rtol=1e-10, maxit=2000)
        np.testing.assert_allclose(X1[:, j].cpu().numpy(), oc["x"], rtol=1e-6, atol=1e-7)
    if k == 1:
        h0, h1 = np.asarray(R0[0].history), np.asarray(R1[0].history)
        m = min(R0[0].iterations, R1[0].iterations) - 5
        assert (h1[:m] > 0).all()
        # both follow one residual, which falls by ten orders of magnitude
        assert np.abs(np.log10(h1[:m]) - np.log10(h0[:m])).max() < 1.0
    cap = R0[0].iterations * 2 // 3
    _, R2 = run(cap, precision="f32-refined")
    assert _resident(A) == 1
    assert max(r.iterations for r in R2) == cap and not R2[0].converged


def test_a_held_chip_costs_a_small_solve_little(cuda):
    """CUs that do not come free are waited for a hundredth of a second."""
    from diploma_research_amd.csr5 import conjugate_gradient_batched

    rp, ci, v = matgen.varcoef((24, 25), 0.5, seed=3)
    n = len(rp) - 1
    b = to_dev(np.random.default_rng(3).uniform(-1, 1, n))
    A = Csr5.from_csr((n, n, rp, ci, v), sigma=8)
    S = Csr5.from_csr_batched([(n, rp, ci, v)], sigma=8)
    for _ in range(2):  # (the first solves also load the kernels)
        _resident(A, NEVER_SEATED)
        _resident(S, NEVER_SEATED)
        _, r = conjugate_gradient(A, b, rtol=1e-10)
        _, (q,) = conjugate_gradient_batched(S, b, rtol=1e-10)
    assert r.converged and r.seconds < 0.3
    assert q.converged and q.seconds < 0.3


def test_solves_of_other_handles_are_not_held_up(cuda):
    """A small solve beside another thread's long one ends before it."""
    import threading
    import time

    import torch

    # about 2 us an iteration, and far more of them than the tolerance needs
    rp, ci, v = matgen.varcoef((520, 520), 2.0, seed=1)
    n = len(rp) - 1
    long = Csr5.from_csr((n, n, rp, ci, v), sigma=8)
    b = to_dev(np.random.default_rng(1).uniform(-1, 1, n))
    rs, cs, vs = matgen.varcoef((40, 41), 0.5, seed=2)
    m = len(rs) - 1
    short = Csr5.from_csr((m, m, rs, cs, vs), sigma=8)
    bs = np.random.default_rng(2).uniform(-1, 1, m)
    conjugate_gradient(short, to_dev(bs), rtol=1e-10)
    conjugate_gradient(long, b, rtol=1e-1, max_iters=5)
    s_long, others = torch.cuda.Stream(), [torch.cuda.Stream() for _ in range(8)]
    bd, marks = to_dev(bs), [torch.zeros(8, device="cuda") for _ in others]
    for mark in marks:  # (loads the kernel)
        mark.add_(1)
    torch.cuda.synchronize()
    ended = {}

    def solve_long():
        conjugate_gradient(long, b, x=torch.zeros_like(b), rtol=1e-200, max_iters=100000, stream=s_long)
        ended["long"] = time.perf_counter()

    t = threading.Thread(target=solve_long)
    x0 = torch.zeros_like(bd)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    t.start()
    time.sleep(0.05)  # (the long solve is on the GPU by then)
    # a stream that does not share the long solve's hardware queue
    events = [torch.cuda.Event() for _ in others]
    for q, e, mark in zip(others, events, marks):
        with torch.cuda.stream(q):
            mark.add_(1)
        e.record(q)
    free = []
    while not free and t.is_alive():
        free = [q for q, e in zip(others, events) if e.query()]
    assert free and t.is_alive()
    x, r = conjugate_gradient(short, bd, x=x0, rtol=1e-10, stream=free[0])
    ended["short"] = time.perf_counter()
    t.join()
    assert r.converged and r.relres_true <= 1.01e-10
    assert ended["long"] - t0 > 0.3, "the long solve is not long"
    assert ended["short"] < ended["long"]
    oc = O.Csr5(m, m, rs, cs, vs).cg(bs, rtol=1e-10, maxit=2000)
    np.testing.assert_allclose(x.cpu().numpy(), oc["x"], rtol=1e-7, atol=1e-8)


@pytest.mark.parametrize("sigma", [5, 16])
def test_called_off_batches_take_the_form_asked_for(cuda, sigma):
    """Where the resident workgroups are not seated, a batch kept by diagonals
    is solved by the launch sequence or, with persistent=True, by the
    cooperative kernel: the same bits."""
    import torch

    from diploma_research_amd.csr5 import conjugate_gradient_batched

    systems = []
    for i, side in enumerate([11, 37, 5, 60, 23, 48]):
        rp, ci, v = matgen.varcoef((side, side), 0.5, seed=i)
        systems.append((side * side, rp, ci, v))
    A = Csr5.from_csr_batched(systems, sigma=sigma)
    b = to_dev(np.random.default_rng(0).uniform(-1, 1, sum(n for n, *_ in systems)))
    got = []
    for persistent in (False, True, True):
        _resident(A, NEVER_SEATED)
        X, R = conjugate_gradient_batched(A, b, rtol=1e-10, max_iters=3000, persistent=persistent)
        assert all(r.converged and r.relres_true <= 1.01e-10 for r in R)
        got.append((X, [r.iterations for r in R]))
    for X, its in got[1:]:
        assert torch.equal(X, got[0][0]) and its == got[0][1]
    assert _resident(A) == 0
    Xr, _ = conjugate_gradient_batched(A, b, rtol=1e-10, max_iters=3000)
    assert _resident(A) == 1
    np.testing.assert_allclose(Xr.cpu().numpy(), got[0][0].cpu().numpy(), rtol=1e-7, atol=1e-8)


# many small systems, which the launch sequence iterates side by side, and a few
# that fill an XCD each
@pytest.mark.parametrize("shape,systems,resident", [((20, 25), 256, 1), ((20, 25), 300, 0), ((60, 70), 200, 0),
                                                    ((300, 310), 20, 1)])
def test_batches_that_would_take_too_many_turns(cuda, shape, systems, resident):
    from diploma_research_amd.csr5 import conjugate_gradient_batched

    rp, ci, v = matgen.varcoef(shape, 0.5, seed=systems)
    n = len(rp) - 1
    A = Csr5.from_csr_batched([(n, rp, ci, v)] * systems, sigma=5)
    x = np.random.default_rng(systems).uniform(-1, 1, (systems, n))
    some = sorted({0, 1, systems // 2, systems - 1})
    b = np.zeros((systems, n))
    for i in range(systems):
        b[i] = O.csr_spmv(rp, ci, v, x[i])
    _resident(A)
    X, R = conjugate_gradient_batched(A, to_dev(b.ravel()), rtol=1e-10, max_iters=5000)
    assert _resident(A) == resident
    assert all(r.converged and r.relres_true <= 1.01e-10 for r in R)
    X = X.cpu().numpy().reshape(systems, n)
    for i in some:
        oc = O.Csr5(n, n, rp, ci, v).cg(b[i], rtol=1e-10, maxit=5000)
        np.testing.assert_allclose(X[i], oc["x"], rtol=1e-6, atol=1e-7)
