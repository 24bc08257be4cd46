"""GPU tests of the batched solve and refinement at the edges of its tiles,
slabs and strips, and of the requests that leave it for the single solve."""
import numpy as np
import pytest
import torch

from oracle import candmc_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def Q():
    from candmc_amd import qr
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    return qr


def problem(m, n, k, kappa, seed):
    """A = orthonormal columns scaled from 1 to 1/kappa, x known, b = A·x + a residual."""
    q = np.linalg.qr(O.gaussian(m, n, seed))[0]
    A = q * np.logspace(0, -np.log10(kappa), n)
    x = O.gaussian(n, k, seed + 1)
    r = O.gaussian(m, k, seed + 2)
    r -= q @ (q.T @ r)
    return A, A @ x + r, x


def pad(Q, A, ld, fill=3.0):
    P = np.full((ld, A.shape[1]), fill)
    P[:A.shape[0]] = A
    return Q.to_gpu(P)


def solve(Q, probs, max_iter=4, tol=1e-12, shared=False):
    reqs, outs, keep = [], [], []
    total = sum(A.shape[1] for A, _, _ in probs)
    width = max(B.shape[1] for _, B, _ in probs)
    common = torch.full((total * width,), 5.0, dtype=torch.float64, device="cuda")
    at = 0
    for A, B, _ in probs:
        m, n, k = *A.shape, B.shape[1]
        dA, dB = pad(Q, A, m + 3), pad(Q, B, m + 1)
        X, ldx = (common[at:], total) if shared else (torch.full(((n + 2) * k,), 5.0, dtype=torch.float64, device="cuda"), n + 2)
        at += n
        keep += [dA, dB]
        outs.append((X, ldx, n, k))
        reqs.append((dA, m + 3, m, n, dB, m + 1, k, X, ldx))
    torch.cuda.synchronize()
    res = Q.lstsq_batched(reqs, max_iter=max_iter, tol=tol)
    xs = []
    for X, ldx, n, k in outs:
        h = X.cpu().numpy()
        xs.append(np.stack([h[j * ldx:j * ldx + n] for j in range(k)], axis=1))
        if not shared:
            assert all((h[j * ldx + n:(j + 1) * ldx] == 5.0).all() for j in range(k))
    return xs, res


# relative error: the last step is below 1e-12 and the fixed point within
# kappa·ε·√(m·n) of the solution, at most 1e2·2.2e-16·√(9000·128) = 2.4e-11
TOL = 3e-11
SIZES = [(1, 1, 1), (5, 3, 16), (15, 15, 2), (128, 16, 1), (129, 17, 3), (127, 33, 16), (255, 48, 5), (64, 64, 4),
         (4099, 64, 7), (385, 65, 15), (1000, 100, 9), (128, 127, 1), (300, 128, 16), (8257, 128, 2), (9000, 12, 8)]


@pytest.mark.parametrize("shared", [False, True])
def test_edges(Q, shared):
    print("lstsq_batched edges, shared", shared, flush=True)
    probs = [problem(m, n, k, 1e2 if n > 1 else 1.0, 7 * m + n) for m, n, k in SIZES]
    xs, res = solve(Q, probs, shared=shared)
    for (m, n, k), (A, B, x), got, r in zip(SIZES, probs, xs, res):
        assert r[0] == 0 and 1 <= r[1] <= 4 and r[2] <= 1e-12, (m, n, k, r)
        assert np.abs(got - x).max() <= TOL * np.abs(x).max(), (m, n, k)


def test_first_solution_alone(Q):
    print("lstsq_batched without refinement", flush=True)
    probs = [problem(m, n, k, 1e2 if n > 1 else 1.0, m + n) for m, n, k in SIZES]
    xs, res = solve(Q, probs, max_iter=0)
    for (m, n, k), (A, B, x), got, r in zip(SIZES, probs, xs, res):
        assert r == (0, 0, 0.0)
        # the factorization's backward error, kappa·m·n·ε at worst
        assert np.abs(got - x).max() <= 1e2 * m * n * 2.3e-16 * np.abs(x).max(), (m, n, k)


def test_requests_that_leave(Q):
    """κ = 1e9 (semi-normal steps do not contract), a NaN entry, and a column
    of zeros among ordinary requests: each ends as it does alone."""
    print("lstsq_batched, requests that leave", flush=True)
    probs = [problem(700, 40, 3, 1e2, 1), problem(700, 40, 3, 1e9, 2), problem(700, 40, 3, 1e2, 3),
             problem(700, 40, 3, 1e2, 4), problem(300, 20, 2, 1e2, 5)]
    probs[2][0][5, 5] = np.nan
    probs[3][0][:, 7] = 0.0
    xs, res = solve(Q, probs, max_iter=8)
    assert res[0][0] == 0 and res[4][0] == 0
    for i in (0, 4):
        assert np.abs(xs[i] - probs[i][2]).max() <= TOL * np.abs(probs[i][2]).max()
    assert res[1][0] in (0, 6) and res[2][0] == 5 and res[3][0] != 0
    for i in range(5):
        x1, r1 = solve(Q, [probs[i]], max_iter=8)
        assert np.array_equal(x1[0], xs[i], equal_nan=True) and r1[0][:2] == res[i][:2]
