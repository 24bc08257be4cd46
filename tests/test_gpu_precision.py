"""GPU tests of accuracy: the error of the FP64 products, factorizations and
solves against the same thing in extended precision, next to the error of a
plain FP64 numpy rendering of the same algorithm on the same inputs.  Both are
rounding errors of a few units; the bound is a small multiple of numpy's, the
mean over several seeds (sums that start from a large value, or long chains of
them, show as more)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
X = np.longdouble
SEEDS = range(6)


@pytest.fixture(scope="module")
def Q():
    from candmc_amd import qr
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    return qr


def rnd(m, n, seed):
    return np.asfortranarray(np.random.default_rng(seed).standard_normal((m, n)))


def err(got, ref):
    e = (got - ref).astype(np.float64)
    return float(np.linalg.norm(e) / np.linalg.norm(ref.astype(np.float64)))


def zeros(n):
    return torch.zeros(n, dtype=torch.float64, device="cuda")


@pytest.mark.parametrize("n,nr", [(512, 3), (600, 1), (600, 16), (1100, 5)])
@pytest.mark.parametrize("trans", [False, True])
def test_triangular_solve(Q, n, nr, trans):
    """The chained solve (four blocks of 128 rows and more): at most twice the
    error of the same block steps in numpy (block inverse, product, subtraction)."""
    ours, plain = [], []
    for seed in SEEDS:
        R = np.triu(rnd(n, n, seed)) / np.sqrt(n) + 2 * np.diag(np.sign(rnd(n, 1, seed + 50)[:, 0]))
        B = rnd(n, nr, seed + 100)
        M = R.T if trans else R
        ref = B.astype(X)
        for i in (range(n) if trans else range(n - 1, -1, -1)):
            ref[i] /= X(M[i, i])
            rest = slice(i + 1, n) if trans else slice(0, i)
            ref[rest] -= np.outer(M[rest, i].astype(X), ref[i])
        Y = B.copy()
        blocks = [(j, min(n, j + 128)) for j in range(0, n, 128)]
        for a, b in (blocks if trans else blocks[::-1]):
            Y[a:b] = np.linalg.inv(M[a:b, a:b]) @ Y[a:b]
            rest = slice(b, n) if trans else slice(0, a)
            Y[rest] -= M[rest, a:b] @ Y[a:b]
        plain.append(err(Y, ref))
        print("trsm", n, nr, trans, seed, flush=True)
        dR, dB = Q.to_gpu(np.asfortranarray(R)), Q.to_gpu(B)
        Q.trsm_r(dR, n, n, dB, n, nr, trans=trans)
        ours.append(err(Q.from_gpu(dB, n, nr), ref))
    assert np.mean(ours) < 2 * np.mean(plain), (np.mean(ours), np.mean(plain))


@pytest.mark.parametrize("m,b", [(256, 32), (256, 128), (130, 100), (500, 64), (1000, 16)])
def test_explicit_q(Q, m, b):
    """construct_Q1 of one leaf from its own V and T, Q1 = [I; 0] − V·(T·V_topᵀ):
    the largest error at most twice that of the same products in numpy."""
    assert Q.plan_tsqr(m, b, 1)[0] == 1
    ours, plain = [], []
    for seed in SEEDS:
        print("construct_Q1", m, b, seed, flush=True)
        dA, R, tau, Q1 = Q.to_gpu(rnd(m, b, seed)), zeros(b * b), zeros(b), zeros(m * b)
        td = zeros(Q.tree_data_size(m, b, 1))
        Q.bitree_tsqr(dA, m, R, tau, m, b, numPes=1, output_Y=1, tree_data=td)
        Q.construct_Q1(dA, m, tau, Q1, m, m, b, b, numPes=1, tree_data=td)
        V = np.tril(Q.from_gpu(dA, m, b), -1) + np.eye(m, b)
        T = np.triu(Q.from_gpu(td[:b * b], b, b))
        E = np.eye(m, b)
        ref = E - V.astype(X) @ (T.astype(X) @ V[:b].T.astype(X))
        ours.append(float(abs(Q.from_gpu(Q1, m, b) - ref).max()))
        plain.append(float(abs(E - V @ (T @ V[:b].T) - ref).max()))
    assert np.mean(ours) < 2 * np.mean(plain), (np.mean(ours), np.mean(plain))


@pytest.mark.parametrize("b", [32, 64, 128])
def test_signed_lu(Q, b):
    """L and U of the signed LU of an orthonormal block against plain
    right-looking elimination in numpy, which rounds an entry at every column
    before it; here the sixteen columns of a strip are one update, which at two
    strips already saves a third of an entry's roundings."""
    ours, plain = [], []
    for seed in SEEDS:
        print("signed LU", b, seed, flush=True)
        A = np.asfortranarray(np.linalg.qr(rnd(512, b, seed))[0][:b])

        def lu(M):
            for j in range(b):
                M[j, j] -= -1 if M[j, j] > 0 else 1
                M[j + 1:, j] /= M[j, j]
                M[j + 1:, j + 1:] -= np.outer(M[j + 1:, j], M[j, j + 1:])
            return M

        ref, P = lu(A.astype(X)), lu(A.copy())
        dA, R = Q.to_gpu(A), zeros(b * b)
        Q.signed_NLU(dA, R, b, b, b)
        G = Q.from_gpu(dA, b, b)
        ours.append([err(np.triu(G), np.triu(ref)), err(np.tril(G, -1), np.tril(ref, -1))])
        plain.append([err(np.triu(P), np.triu(ref)), err(np.tril(P, -1), np.tril(ref, -1))])
    u, p = np.mean(ours, 0), np.mean(plain, 0)
    assert u[0] < 0.75 * p[0] and u[1] < p[1], (u, p)


@pytest.mark.parametrize("m,b", [(256, 32), (256, 64), (256, 128)])
def test_leaf_r(Q, m, b):
    """R of one leaf against plain column by column elimination in numpy, which
    rounds twice (product, sum) where the leaf's products round once: an error
    below 0.88 of numpy's, if the sums over the rows are no long chains."""
    def r_of(A):
        A = A.copy()
        for j in range(b):
            x = A[j:, j].copy()
            beta = -np.copysign(np.sqrt((x * x).sum()), x[0])
            v, tau = x / (x[0] - beta), (beta - x[0]) / beta
            v[0] = 1
            A[j:, j + 1:] -= tau * np.outer(v, v @ A[j:, j + 1:])
            A[j, j], A[j + 1:, j] = beta, 0
        return A[:b]

    ours, plain = [], []
    for seed in SEEDS:
        print("leaf", m, b, seed, flush=True)
        A = rnd(m, b, seed)
        ref = r_of(A.astype(X))
        dA, T = Q.to_gpu(A), zeros(b * b)
        Q.local_tsqr(dA, T, m, b, m)
        ours.append(err(np.triu(Q.from_gpu(dA, m, b)[:b]), ref))
        plain.append(err(r_of(A), ref))
    assert np.mean(ours) < 0.88 * np.mean(plain), (np.mean(ours), np.mean(plain))


@pytest.mark.parametrize("k", [128, 256])
def test_small_product(Q, k):
    """Y1ᵀ·Y2 of positive entries (sums that only grow): at most 1.35 times the
    error of four running FP64 sums added up at the end."""
    ours, plain = [], []
    for seed in SEEDS:
        print("small product", k, seed, flush=True)
        A, B = np.abs(rnd(k, 32, seed)), np.abs(rnd(k, 32, seed + 9))
        ref = A.T.astype(X) @ B.astype(X)
        sums = [np.zeros((32, 32)) for _ in range(4)]
        for i in range(k):
            j = i // 4 % 4
            sums[j] = (sums[j].astype(X) + np.outer(A[i].astype(X), B[i].astype(X))).astype(np.float64)
        plain.append(err((sums[0] + sums[1]) + (sums[2] + sums[3]), ref))
        dT = zeros(32 * 32)
        Q.compute_invT_from_Y2(Q.to_gpu(np.asfortranarray(A)), k, Q.to_gpu(np.asfortranarray(B)), k, dT, 32, k, 32, 32)
        ours.append(err(Q.from_gpu(dT, 32, 32), ref))
    assert np.mean(ours) < 1.35 * np.mean(plain), (np.mean(ours), np.mean(plain))
