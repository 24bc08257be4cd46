"""GPU test of the one-launch blocked triangular solve at the edges of its
blocks and tiles (from 385 columns on), against a solve in extended
precision, with odd leading dimensions."""
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


@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("n,nrhs", [(385, 1), (400, 16), (512, 4), (513, 3), (527, 15), (640, 2), (1100, 5), (1921, 16)])
def test_trsm(Q, n, nrhs, trans):
    print("trsm chain", n, nrhs, trans, flush=True)
    # unit-scale diagonal and small off-diagonal entries: condition about 3
    R = np.triu(O.gaussian(n, n, n)) / (2.0 * n) + np.diag(1.0 + 0.5 * np.sin(np.arange(n)))
    X = O.gaussian(n, nrhs, n + 1)
    M = R.T if trans else R
    Bx = (M.astype(np.longdouble) @ X.astype(np.longdouble)).astype(np.float64)
    A = np.full((n + 3, n), 5.0)                    # below the diagonal: not R's
    A[:n] = R + np.tril(np.full((n, n), 5.0), -1)
    P = np.full((n + 1, nrhs), 7.0)
    P[:n] = Bx
    dB = Q.to_gpu(P)
    Q.trsm_r(Q.to_gpu(A), n + 3, n, dB, n + 1, nrhs, trans=trans)
    got = Q.from_gpu(dB, n + 1, nrhs)
    assert (got[n:] == 7.0).all()
    # condition 3, n-term sums in the blocks and their inverses
    assert np.abs(got[:n] - X).max() <= 3 * 4 * n * np.finfo(np.float64).eps * np.abs(X).max()
