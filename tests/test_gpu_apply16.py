"""GPU tests of the implicit TSQR Q's panel-by-panel application at the edges
of its tiles, strips and leaf sizes, with odd leading dimensions."""
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


def padded(A, ld):
    P = np.full((ld, A.shape[1]), 7.0)
    P[:A.shape[0]] = A
    return P


def factor(Q, A, P):
    m, b = A.shape
    L, _, _ = Q.plan_tsqr(m, b, P)
    dY = Q.to_gpu(padded(A, m + 1))
    dR = torch.zeros(b * b, dtype=torch.float64, device="cuda")
    dtau = torch.zeros(L * b, dtype=torch.float64, device="cuda")
    td = torch.zeros(Q.tree_data_size(m, b, P), dtype=torch.float64, device="cuda")
    Q.bitree_tsqr(dY, m + 1, dR, dtau, m, b, numPes=P, output_Y=1, tree_data=td)

    def apply(B, trans):
        k = B.shape[1]
        dB = Q.to_gpu(padded(B, m + 3))
        Q.apply_tsqr_QT(dY, m + 1, dtau, dB, m + 3, m, b, k, numPes=P, tree_data=td, trans=trans)
        got = Q.from_gpu(dB, m + 3, k)
        assert (got[m:] == 7.0).all()
        return got[:m]
    return Q.from_gpu(dY, m + 1, b)[:m], dtau.cpu().numpy(), Q.from_gpu(dR, b, b), apply


@pytest.mark.parametrize("m,b,k", [(1, 1, 1), (16, 15, 16), (17, 16, 17), (127, 33, 63), (128, 127, 65), (129, 128, 64),
                                   (241, 65, 15), (256, 17, 130), (257, 32, 3), (300, 48, 64), (511, 64, 33),
                                   (512, 16, 5), (513, 16, 20)])
def test_one_leaf_against_reflectors(Q, m, b, k):
    print("one leaf", m, b, k, flush=True)
    Y, tau, _, apply = factor(Q, O.gaussian(m, b, m + b), 1)
    V = np.tril(Y, -1) + np.eye(m, b)
    B = O.gaussian(m, k, k)
    want = B.copy()
    for i in range(b):
        want -= tau[i] * np.outer(V[:, i], V[:, i] @ want)
    # both sides apply b reflectors whose products have m terms
    tol = 4 * b * np.sqrt(m) * EPS * np.linalg.norm(B, axis=0) + EPS
    got = apply(B, True)
    assert (np.linalg.norm(got - want, axis=0) <= tol).all()
    assert (np.linalg.norm(apply(got, False) - B, axis=0) <= tol).all()


@pytest.mark.parametrize("m,b,P,k", [(2, 1, 2, 1), (50, 16, 3, 16), (90, 17, 5, 70), (1000, 100, 7, 129),
                                     (1285, 128, 10, 31), (3000, 63, 0, 65), (700, 127, 4, 64)])
def test_tree(Q, m, b, P, k):
    print("tree", m, b, P, k, flush=True)
    A = O.gaussian(m, b, m + b)
    _, _, R, apply = factor(Q, A, P)
    levels = 8
    z = np.zeros((m, b))
    z[:b] = R
    tol = 4 * levels * b * np.sqrt(m) * EPS
    assert (np.linalg.norm(apply(A, True) - z, axis=0) <= tol * np.linalg.norm(A, axis=0)).all()
    B = O.gaussian(m, k, k)
    back = apply(apply(B, True), False)
    assert (np.linalg.norm(back - B, axis=0) <= tol * np.linalg.norm(B, axis=0)).all()
