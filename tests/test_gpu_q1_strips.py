"""GPU test of construct_Q1 at the edges of its 16-column strips and their
pairs: Q1 orthonormal and Q1·R = A, with odd leading dimensions."""
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


@pytest.mark.parametrize("m,b,P", [(1, 1, 1), (33, 15, 2), (16, 16, 1), (90, 17, 5), (700, 31, 3), (1000, 32, 6),
                                   (555, 33, 4), (900, 48, 9), (2100, 64, 8), (513, 65, 3), (1285, 80, 10),
                                   (4099, 100, 0), (1500, 113, 7), (1397, 127, 11), (2561, 128, 13)])
def test_explicit_q(Q, m, b, P):
    print("construct_Q1", m, b, P, flush=True)
    A = O.gaussian(m, b, m + b)
    Ap = np.full((m + 1, b), 7.0)
    Ap[:m] = A
    L, _, _ = Q.plan_tsqr(m, b, P)
    dY = Q.to_gpu(Ap)
    dR = torch.zeros(b * b, dtype=torch.float64, device="cuda")
    dtau = torch.zeros(L * b, dtype=torch.float64, device="cuda")
    td = torch.zeros(Q.tree_data_size(m, b, P), dtype=torch.float64, device="cuda")
    Q.bitree_tsqr(dY, m + 1, dR, dtau, m, b, numPes=P, output_Y=1, tree_data=td)
    dQ = Q.to_gpu(np.full((m + 3, b), 7.0))
    Q.construct_Q1(dY, m + 1, dtau, dQ, m + 3, m, b, b, numPes=P, tree_data=td)
    got = Q.from_gpu(dQ, m + 3, b)
    assert (got[m:] == 7.0).all()
    got, R = got[:m], Q.from_gpu(dR, b, b)
    # b reflectors in a leaf and in each of at most five levels, columnwise
    tol = 4 * 6 * b * np.sqrt(m) * EPS
    assert (np.linalg.norm(got.T @ got - np.eye(b), axis=0) <= tol).all()
    assert (np.linalg.norm(got @ R - A, axis=0) <= tol * np.linalg.norm(A, axis=0)).all()
