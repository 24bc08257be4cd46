"""GPU tests of the sixteen-column panel kernels (leaf QR of more than 64
columns, every tree node): tile edges in rows and columns, and inputs that
leave the fast range of the column step (zero, tiny, huge and non-finite
columns), against LAPACK dgeqrf and the factorization's own identities.

Tolerance: Householder QR is columnwise backward stable with a constant
proportional to the number of rows; 64·m·ε relative to each column's norm."""
import numpy as np
import pytest
import torch

from oracle import candmc_oracle as O

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


@pytest.fixture(scope="module")
def Q():
    from candmc_amd import qr
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    return qr


def matrix(kind, m, b, seed):
    A = O.gaussian(m, b, seed)
    rng = np.random.default_rng(seed)
    if kind == "zero":
        A[:, [0, b // 2, b - 1]] = 0.0
    elif kind == "scaled":                       # each column its own scale, 1e-250 .. 1e250
        A *= 10.0 ** rng.uniform(-250, 250, b)
    elif kind == "tiny":
        A *= 1e-300
    elif kind == "huge":
        A *= 1e300
    return np.asfortranarray(A)


def colmax(E, A):
    """Largest column norm of E relative to A's (each scaled to avoid overflow)."""
    s = np.abs(A).max(0)
    s[s == 0] = 1.0
    n = np.linalg.norm(A / s, axis=0)
    return float((np.linalg.norm(E / s, axis=0) / np.where(n > 0, n, 1.0)).max())


def leaf(Q, A):
    m, b = A.shape
    print("leaf", m, b, flush=True)
    dA, dT = Q.to_gpu(A), torch.zeros(b * b, dtype=torch.float64, device="cuda")
    tau = Q.local_tsqr(dA, dT, m, b, m)
    return Q.from_gpu(dA, m, b), Q.from_gpu(dT, b, b), tau.cpu().numpy()


@pytest.mark.parametrize("m,b,kind", [
    (256, 128, "gauss"), (255, 128, "gauss"), (241, 113, "gauss"), (240, 112, "gauss"), (193, 127, "gauss"),
    (129, 66, "gauss"), (128, 128, "gauss"), (127, 65, "gauss"), (113, 96, "gauss"), (81, 81, "gauss"), (65, 65, "gauss"),
    (256, 128, "zero"), (200, 100, "zero"), (256, 128, "scaled"), (100, 80, "scaled"), (256, 128, "tiny"),
    (130, 70, "tiny"), (256, 128, "huge")])
def test_leaf(Q, m, b, kind):
    A = matrix(kind, m, b, m + b)
    YR, T, tau = leaf(Q, A)
    ref, rtau = O.local_tsqr(A)
    tol = 64 * m * EPS
    assert colmax(np.triu(YR[:b]) - np.triu(ref[:b]), np.triu(ref[:b])) < tol
    assert np.abs(np.tril(YR, -1) - np.tril(ref, -1)).max() < tol * b          # vectors: entries at most 1
    assert np.abs(tau - rtau[:b]).max() < tol and np.array_equal(np.diag(T), tau)
    Y = np.tril(YR, -1)[:, :b] + np.eye(m, b)
    G = Y.T @ Y                                                                # T⁻ᵀ + T⁻¹ = YᵀY
    assert np.abs(T + T.T - T @ G @ T.T).max() < tol and np.array_equal(T, np.triu(T))


def test_leaf_nan_stays_behind_its_column(Q):
    """Columns before a NaN are those of the matrix without it."""
    m, b, j = 256, 128, 41
    A = matrix("gauss", m, b, 3)
    ref, rtau = O.local_tsqr(A)
    A[100, j] = np.nan
    YR, T, tau = leaf(Q, A)
    assert np.abs(YR[:, :j] - ref[:, :j]).max() < 64 * m * EPS * np.abs(ref).max()
    assert np.abs(tau[:j] - rtau[:j]).max() < 64 * m * EPS
    assert np.isnan(YR[:, j]).any()


@pytest.mark.parametrize("m,b,P,kind", [
    (60, 1, 3, "gauss"), (400, 15, 5, "gauss"), (400, 16, 5, "gauss"), (400, 17, 5, "gauss"), (700, 31, 3, "gauss"),
    (700, 33, 3, "gauss"), (900, 48, 7, "gauss"), (900, 49, 2, "gauss"), (1000, 64, 6, "gauss"), (1000, 65, 5, "gauss"),
    (1000, 97, 9, "gauss"), (1300, 113, 11, "gauss"), (1100, 128, 8, "gauss"), (2500, 128, 0, "gauss"),
    (700, 32, 3, "zero"), (1100, 128, 7, "zero"), (700, 30, 3, "scaled"), (1100, 128, 5, "scaled"), (900, 80, 4, "tiny"),
    (900, 64, 4, "huge")])
def test_tree(Q, m, b, P, kind):
    """Q1·R = A and Q1ᵀQ1 = I for the explicit Q of the tree, R upper."""
    print("tree", m, b, P, kind, flush=True)
    A = matrix(kind, m, b, m + b)
    L, _, _ = Q.plan_tsqr(m, b, P)
    dA = Q.to_gpu(A)
    dR = torch.zeros(b * b, dtype=torch.float64, device="cuda")
    tau = torch.zeros(L * b, dtype=torch.float64, device="cuda")
    td = torch.zeros(Q.tree_data_size(m, b, P), dtype=torch.float64, device="cuda")
    Q.bitree_tsqr(dA, m, dR, tau, m, b, numPes=P, output_Y=1, tree_data=td)
    R = Q.from_gpu(dR, b, b)
    dQ = torch.zeros(m * b, dtype=torch.float64, device="cuda")
    Q.construct_Q1(dA, m, tau, dQ, m, m, b, b, numPes=P, tree_data=td)
    Q1 = Q.from_gpu(dQ, m, b)
    tol = 64 * m * EPS
    s = np.abs(A).max(0)
    s[s == 0] = 1.0                                                            # products on scaled columns
    assert np.array_equal(R, np.triu(R))
    assert colmax(Q1 @ (R / s) - A / s, A / s) < tol
    assert np.abs(Q1.T @ Q1 - np.eye(b)).max() < tol
