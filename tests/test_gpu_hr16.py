"""GPU tests of the Householder reconstruction core at the edges of its
16-column strips: the signed LU against its own recurrence, and T, T⁻ᵀ, W
against the identities that define them (one launch forms them all)."""
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


def signed_lu(A):
    """LU of A − S without pivoting, s_i = −1 if pivot i is positive, else +1."""
    M, b = A.copy(), A.shape[0]
    s = np.ones(b)
    with np.errstate(all="ignore"):
        for i in range(b):
            s[i] = -1.0 if M[i, i] > 0 else 1.0
            M[i, i] -= s[i]
            M[i + 1:, i] *= 1.0 / M[i, i]
            M[i + 1:, i + 1:] -= np.outer(M[i + 1:, i], M[i, i + 1:])
    return M, s


def run_nlu(Q, A, R):
    b = A.shape[0]
    print("signed_NLU", b, flush=True)
    dA, dR = Q.to_gpu(A), Q.to_gpu(R)
    sg = torch.zeros(b, dtype=torch.int64, device="cuda")
    Q.signed_NLU(dA, dR, b, b, b, sg)
    return Q.from_gpu(dA, b, b), Q.from_gpu(dR, b, b), sg.cpu().numpy()


EDGES = [1, 2, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 80, 97, 112, 113, 127, 128]


@pytest.mark.parametrize("b", EDGES)
def test_signed_lu(Q, b):
    A = np.linalg.qr(O.gaussian(3 * b + 1, b, b))[0][:b].copy()
    R = np.triu(O.gaussian(b, b, b + 1))
    LU, Rg, s = run_nlu(Q, A, R)
    ref, rs = signed_lu(A)
    assert np.array_equal(s, rs.astype(int)) and np.array_equal(Rg, rs[:, None] * R)
    L, U = np.tril(LU, -1) + np.eye(b), np.triu(LU)
    # backward error of LU: 2·b·ε·|L|·|U| entrywise
    assert (np.abs(L @ U - (A - np.diag(rs))) <= 2 * b * EPS * (np.abs(L) @ np.abs(U)) + 4 * EPS).all()


@pytest.mark.parametrize("b,what", [(100, np.nan), (100, np.inf), (40, np.nan), (90, 1e308)])
def test_signed_lu_extremes(Q, b, what):
    """Columns before a NaN or infinity keep their values; a pivot of 1e308
    scales its column by its true reciprocal."""
    A = np.linalg.qr(O.gaussian(3 * b, b, b))[0][:b].copy()
    j = b // 2 + 3
    A[j, j] = what
    LU, _, _ = run_nlu(Q, A, np.triu(A))
    ref, _ = signed_lu(A)
    assert np.abs(LU[:, :j] - ref[:, :j]).max() < 1e-12
    if np.isfinite(what):
        assert np.allclose(LU[j + 1:, j], ref[j + 1:, j], rtol=1e-10, atol=0) and np.isfinite(LU).all()


@pytest.mark.parametrize("b", EDGES)
def test_reconstruction_factors(Q, b):
    m = 3 * b + 5
    A = O.gaussian(m, b, 900 + b)
    print("hh_recon", m, b, flush=True)
    dA = Q.to_gpu(A)
    W, T, Ti = (torch.full((b * b,), 7.0, dtype=torch.float64, device="cuda") for _ in range(3))
    Q.hh_recon_qr(dA, m, m, b, W, T=T, invT_T=Ti)
    YR, W, T, Ti = Q.from_gpu(dA, m, b), Q.from_gpu(W, b, b), Q.from_gpu(T, b, b), Q.from_gpu(Ti, b, b)
    ref, tau = O.local_tsqr(A)
    tol = 64 * m * EPS
    Y = np.tril(YR, -1)[:, :b] + np.eye(m, b)
    for M, tri in ((W, np.triu), (T, np.triu), (Ti, np.tril)):
        assert np.array_equal(M, tri(M))
    assert np.abs(np.diag(T) - tau[:b]).max() < tol
    assert np.abs(YR - ref).max() < tol * np.abs(ref).max()
    assert np.abs(W + T @ Y[:b].T).max() < tol                          # W = −T·Y1ᵀ
    assert np.abs(Ti @ T.T - np.eye(b)).max() < tol * b                 # T⁻ᵀ·Tᵀ = I
    assert np.abs(T + T.T - T @ (Y.T @ Y) @ T.T).max() < tol            # Q orthogonal
