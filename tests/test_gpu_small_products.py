"""GPU test of the small products at the edges of their tiles: the blocked
solve below four blocks (few columns, both operands' masks) and the Q
application's b×b products with few and with many columns."""
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


@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("n,nrhs", [(1, 1), (15, 16), (16, 2), (17, 5), (64, 1), (100, 16), (127, 3), (128, 4), (129, 15),
                                    (200, 17), (383, 5)])
def test_short_solve(Q, n, nrhs, trans):
    print("short solve", n, nrhs, trans, flush=True)
    R = np.triu(O.gaussian(n, n, n)) / (2.0 * n) + np.diag(1.0 + 0.5 * np.sin(np.arange(n)))
    X = O.gaussian(n, nrhs, n + 1)
    Bx = (R.T if trans else R) @ X
    A = R + np.tril(np.full((n, n), 5.0), -1)
    dB = Q.to_gpu(Bx)
    Q.trsm_r(Q.to_gpu(A), n, n, dB, n, nrhs, trans=trans)
    # condition 3; B itself is rounded to n·ε
    assert np.abs(Q.from_gpu(dB, n, nrhs) - X).max() <= 3 * 8 * n * EPS * max(1.0, np.abs(X).max())


@pytest.mark.parametrize("m,n,b,nrhs", [(200, 33, 16, 1), (200, 33, 16, 17), (300, 100, 100, 5), (300, 100, 100, 40),
                                        (260, 129, 128, 16), (260, 129, 128, 33), (161, 96, 32, 15), (161, 96, 32, 64)])
def test_q_application(Q, m, n, b, nrhs):
    print("Q application", m, n, b, nrhs, flush=True)
    A = O.gaussian(m, n, m + n)
    dA = Q.to_gpu(A)
    Tt = Q.geqrf2d(dA, m, m, n, b)
    YR = Q.from_gpu(dA, m, n)
    B = O.gaussian(m, nrhs, nrhs)
    dB = Q.to_gpu(B)
    Q.apply_qt(dA, m, Tt, m, n, b, dB, m, nrhs, trans=True)
    # n reflectors on both sides, sums of m terms
    tol = 4 * n * np.sqrt(m) * EPS * np.linalg.norm(B, axis=0)
    assert (np.linalg.norm(Q.from_gpu(dB, m, nrhs) - O.apply_QT(YR, B), axis=0) <= tol).all()
    Q.apply_qt(dA, m, Tt, m, n, b, dB, m, nrhs, trans=False)
    assert (np.linalg.norm(Q.from_gpu(dB, m, nrhs) - B, axis=0) <= tol).all()
