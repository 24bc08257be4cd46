"""GPU tests of the leaf QR of at most 64 columns at the edges of its tiles and
of the parts a tall leaf is shared out in (256 rows each), with inputs that
leave the fast range of the column step.  Helpers and tolerance (64·m·ε,
columnwise) as in test_gpu_panel16.py."""
import numpy as np
import pytest

from oracle import candmc_oracle as O
from test_gpu_panel16 import EPS, Q, colmax, leaf, matrix  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,b,kind", [
    (1, 1, "gauss"), (16, 16, "gauss"), (17, 15, "gauss"), (128, 1, "gauss"), (129, 16, "gauss"), (256, 16, "gauss"),
    (256, 17, "gauss"), (160, 32, "gauss"), (33, 33, "gauss"), (255, 48, "gauss"), (64, 64, "gauss"), (256, 64, "gauss"),
    (257, 1, "gauss"), (257, 64, "gauss"), (273, 16, "gauss"), (511, 33, "gauss"), (512, 64, "gauss"), (500, 49, "gauss"),
    (512, 32, "gauss"), (400, 17, "gauss"), (512, 15, "gauss"), (513, 16, "gauss"), (769, 32, "gauss"), (1023, 31, "gauss"),
    (1024, 32, "gauss"), (1024, 7, "gauss"), (256, 64, "zero"), (512, 64, "zero"), (1024, 32, "zero"), (200, 30, "scaled"),
    (512, 64, "scaled"), (900, 16, "scaled"), (512, 50, "tiny"), (1000, 20, "tiny"), (512, 64, "huge"), (1024, 32, "huge")])
def test_leaf(Q, m, b, kind):
    A = matrix(kind, m, b, m + b)
    YR, T, tau = leaf(Q, A)
    ref, rtau = O.local_tsqr(A)
    tol = 64 * m * EPS
    assert colmax(np.triu(YR[:b]) - np.triu(ref[:b]), np.triu(ref[:b])) < tol
    assert np.abs(np.tril(YR, -1) - np.tril(ref, -1)).max() < tol * b
    assert np.abs(tau - rtau[:b]).max() < tol and np.array_equal(np.diag(T), tau)
    Y = np.tril(YR, -1)[:, :b] + np.eye(m, b)
    G = Y.T @ Y
    assert np.abs(T + T.T - T @ G @ T.T).max() < tol and np.array_equal(T, np.triu(T))


@pytest.mark.parametrize("m,b,row", [(512, 64, 100), (512, 64, 400), (1024, 32, 800), (256, 48, 200)])
def test_nan_stays_behind_its_column(Q, m, b, row):
    A = matrix("gauss", m, b, 3)
    j = b // 2 + 1
    ref, rtau = O.local_tsqr(A)
    A[row, j] = np.nan
    YR, T, tau = leaf(Q, A)
    assert np.abs(YR[:, :j] - ref[:, :j]).max() < 64 * m * EPS * np.abs(ref).max()
    assert np.abs(tau[:j] - rtau[:j]).max() < 64 * m * EPS
    assert np.isnan(YR[:, j]).any()
