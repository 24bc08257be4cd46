"""GPU tests of the sixteen-column panels on inputs at the ends of the column
step's range: they take the straight-line steps too (same bits as without the
odd columns, or with the columns scaled by powers of two), or agree with LAPACK
where the columns have to be rescaled."""
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


def leaf(Q, A):
    m, b = A.shape
    print("leaf", m, b, flush=True)
    dA, dT = Q.to_gpu(np.asfortranarray(A)), torch.zeros(b * b, dtype=torch.float64, device="cuda")
    tau = Q.local_tsqr(dA, dT, m, b, m)
    return Q.from_gpu(dA, m, b), Q.from_gpu(dT, b, b), tau.cpu().numpy()


def tree_r(Q, A, P):
    m, b = A.shape
    print("tree", m, b, P, flush=True)
    L, _, _ = Q.plan_tsqr(m, b, P)
    dA, dR = Q.to_gpu(np.asfortranarray(A)), torch.zeros(b * b, dtype=torch.float64, device="cuda")
    tau = torch.zeros(L * b, dtype=torch.float64, device="cuda")
    td = torch.zeros(Q.tree_data_size(m, b, P), dtype=torch.float64, device="cuda")
    Q.bitree_tsqr(dA, m, dR, tau, m, b, numPes=P, output_Y=1, tree_data=td)
    return Q.from_gpu(dR, b, b)


# leaves of one wave a strip, and tall ones of two and four
LEAVES = [(256, 16), (100, 16), (200, 32), (256, 64), (256, 128), (130, 112), (500, 16), (1000, 16), (512, 64), (1000, 32)]


@pytest.mark.parametrize("m,b", LEAVES)
def test_zero_columns_leave_the_others_alone(Q, m, b):
    """The columns before a padding of zeros: bit for bit those of the matrix
    without it; the padding itself is H = I with R = 0."""
    k = b - 4
    A = np.zeros((m, b))
    A[:, :k] = O.gaussian(m, k, m + b)
    YR, T, tau = leaf(Q, A)
    ref, rT, rtau = leaf(Q, A[:, :k])
    assert np.array_equal(YR[:, :k], ref) and np.array_equal(tau[:k], rtau) and np.array_equal(T[:k, :k], rT)
    assert not YR[:, k:].any() and not tau[k:].any() and not T[:, k:].any()


@pytest.mark.parametrize("b", [16, 64, 128])
def test_square_leaf(Q, b):
    """Nothing lies below the last column of b rows: the others as without it."""
    A = O.gaussian(b, b, b)
    YR, T, tau = leaf(Q, A)
    ref, rT, rtau = leaf(Q, A[:, :b - 1])
    assert np.array_equal(YR[:, :b - 1], ref) and np.array_equal(tau[:b - 1], rtau) and tau[b - 1] == 0.0
    want, _ = O.local_tsqr(A)
    assert abs(YR[b - 1, b - 1] - want[b - 1, b - 1]) < 64 * b * EPS * np.abs(want).max()


@pytest.mark.parametrize("m,b,P", [(512, 16, 4), (1000, 32, 8), (600, 64, 3), (1300, 128, 5), (2000, 100, 0)])
def test_zero_columns_in_the_tree(Q, m, b, P):
    k = b - 4
    A = np.zeros((m, b))
    A[:, :k] = O.gaussian(m, k, m + b)
    L, _, _ = Q.plan_tsqr(m, b, P)
    R, ref = tree_r(Q, A, L), tree_r(Q, A[:, :k], L)
    assert np.array_equal(R[:k, :k], ref) and not R[:, k:].any()


@pytest.mark.parametrize("m,b,row", [(256, 16, 200), (256, 16, 9), (500, 16, 400), (1000, 16, 900), (1000, 32, 700), (512, 64, 300)])
def test_entries_too_small_to_square(Q, m, b, row):
    """A column of one large entry on the diagonal and one of 1e-200 below it
    is no zero column: dlarfg reflects it (tau = 2 or 0 turns on a nonzero x)."""
    A = O.gaussian(m, b, m + b)
    A[:, 5] = 0.0
    A[5, 5], A[row, 5] = 1.0, 1e-200
    A[:5, :5] = np.triu(A[:5, :5])     # the first five columns leave column 5 as it is
    A[5:, :5] = 0.0
    YR, T, tau = leaf(Q, A)
    ref, rtau = O.local_tsqr(np.asfortranarray(A))
    assert np.abs(tau - rtau[:b]).max() < 64 * m * EPS
    assert np.abs(np.triu(YR[:b]) - np.triu(ref[:b])).max() < 64 * m * EPS * np.abs(ref).max()


@pytest.mark.parametrize("e", [-470, -300, 300, 470])
@pytest.mark.parametrize("m,b", LEAVES)
def test_scaled_leaf(Q, m, b, e):
    """A·2^e (entries 1e±141 and 1e±90) takes the same steps: the same
    reflectors, R scaled exactly."""
    A = O.gaussian(m, b, m + b)
    YR, T, tau = leaf(Q, A)
    YS, TS, ts = leaf(Q, np.ldexp(A, e))
    assert np.array_equal(T, TS) and np.array_equal(tau, ts)
    assert np.array_equal(np.tril(YR, -1), np.tril(YS, -1))
    assert np.array_equal(np.ldexp(np.triu(YR[:b]), e), np.triu(YS[:b]))


@pytest.mark.parametrize("e", [-470, 300])
@pytest.mark.parametrize("m,b,P", [(512, 16, 4), (600, 64, 3), (1300, 128, 5), (2000, 100, 0)])
def test_scaled_tree(Q, m, b, P, e):
    A = O.gaussian(m, b, m + b)
    assert np.array_equal(np.ldexp(tree_r(Q, A, P), e), tree_r(Q, np.ldexp(A, e), P))


@pytest.mark.parametrize("m,b", [(256, 16), (256, 128), (512, 64)])
def test_one_scaled_column(Q, m, b):
    """A column of 1e±120 among ordinary ones: its own entries of R scaled, all
    else the same."""
    A = O.gaussian(m, b, m + b)
    d = np.ones(b)
    d[[3, b - 2]] = 2.0 ** -400, 2.0 ** 400
    YR, T, tau = leaf(Q, A)
    YS, TS, ts = leaf(Q, A * d)
    assert np.array_equal(T, TS) and np.array_equal(tau, ts)
    assert np.array_equal(np.tril(YR, -1), np.tril(YS, -1))
    assert np.array_equal(np.triu(YR[:b]) * d, np.triu(YS[:b]))


@pytest.mark.parametrize("m,b", [(256, 16), (65536, 16), (8192, 64), (32768, 128)])
@pytest.mark.parametrize("kind", ["1e-200", "1e200", "nan"])
def test_general_route_is_not_much_slower(Q, m, b, kind):
    """Panels that have to be redone column by column: at most four times an
    ordinary panel's time (three to five passes over a strip in place of two,
    serial loads in place of none; through memory it was five to twenty-four)."""
    print("general route", m, b, kind, flush=True)
    A = Q.to_gpu(O.gaussian(m, b, m + b))
    Z = A.clone()
    if kind == "nan":
        Z[5 * m + 7] = float("nan")
    else:
        Z *= float(kind)
    W = torch.zeros(b * b, dtype=torch.float64, device="cuda")
    work = torch.empty_like(A)

    def us(src):
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        ts = []
        for _ in range(9):
            work.copy_(src)
            torch.cuda.synchronize()
            ev[0].record()
            Q.hh_recon_qr(work, m, m, b, W, numPes=0, sync=False)
            ev[1].record()
            torch.cuda.synchronize()
            ts.append(ev[0].elapsed_time(ev[1]))
        return sorted(ts)[4]

    us(A)
    assert us(Z) < 4 * us(A)


@pytest.mark.parametrize("e", [-474, 505])
@pytest.mark.parametrize("m,b", LEAVES)
def test_scaled_to_the_ends(Q, m, b, e):
    """As far as a column's ‖x‖² neither falls below 2^-960 nor overflows."""
    A = O.gaussian(m, b, m + b)
    YR, T, tau = leaf(Q, A)
    YS, TS, ts = leaf(Q, np.ldexp(A, e))
    assert np.array_equal(T, TS) and np.array_equal(tau, ts)
    assert np.array_equal(np.tril(YR, -1), np.tril(YS, -1))
    assert np.array_equal(np.ldexp(np.triu(YR[:b]), e), np.triu(YS[:b]))


@pytest.mark.parametrize("e", [-560, 509, 700])
@pytest.mark.parametrize("m,b", [(256, 16), (256, 128), (512, 64), (1000, 16)])
def test_one_column_past_the_ends(Q, m, b, e):
    """A column whose ‖x‖² underflows or overflows sends its strip the general
    way; the result is that of the unscaled matrix to rounding."""
    A = O.gaussian(m, b, m + b)
    d = np.zeros(b, int)
    d[b - 3] = e
    YR, T, tau = leaf(Q, A)
    YS, TS, ts = leaf(Q, np.ldexp(A, d))
    tol = 64 * m * EPS
    assert np.abs(T - TS).max() < tol * b and np.abs(tau - ts).max() < tol
    assert np.abs(np.tril(YR, -1) - np.tril(YS, -1)).max() < tol * b
    assert np.abs(np.triu(YR[:b]) - np.ldexp(np.triu(YS[:b]), -d)).max() < tol * np.abs(YR[:b]).max()
