"""GPU test of batched least squares whose partial sums do not fit the arena
at once (many widths: a factorization group is one width, the sums are all of
them): the requests are then solved in several chunks."""
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


def test_chunks(Q):
    """Every request as it is alone, bit for bit, among them one with a NaN and
    one too ill-conditioned for the batched steps, both in the first chunk and
    so taken by the single solve while later chunks are still to come."""
    m, widths, k = 640, list(range(8, 126)), 16
    print("lstsq_batched in chunks", len(widths), flush=True)
    probs = []
    for n in widths:
        A, B = O.gaussian(m, n, 3 * n), O.gaussian(m, k, 3 * n + 1)
        if n == 11:
            A[5, 2] = np.nan
        if n == 13:
            A = np.linalg.qr(A)[0] * np.logspace(0, -9, n)
        probs.append((A, B))
    dev = [(Q.to_gpu(np.asfortranarray(A)), Q.to_gpu(B)) for A, B in probs]

    def solve(idx):
        X = [torch.full((widths[i] * k,), 5.0, dtype=torch.float64, device="cuda") for i in idx]
        reqs = [(dev[i][0], m, m, widths[i], dev[i][1], m, k, x, widths[i]) for i, x in zip(idx, X)]
        res = Q.lstsq_batched(reqs, max_iter=8, tol=1e-12)
        return reqs, [Q.from_gpu(x, widths[i], k) for i, x in zip(idx, X)], res

    reqs, xs, res = solve(range(len(widths)))
    # more partial sums (m/128 slabs a request) than the arena has beside A and T
    room = Q.lstsq_batched_workspace_bytes(reqs) - 8 * sum(m * n + n * n for n in widths)
    assert sum(8 * (m // 128) * n * k for n in widths) > room
    for i, n in enumerate(widths):
        if n in (11, 13):
            continue
        assert res[i][0] == 0 and res[i][2] <= 1e-12
        want = np.linalg.lstsq(*probs[i], rcond=None)[0]
        # κ below 10 for these shapes: a few hundred roundings
        assert np.abs(xs[i] - want).max() <= 1e-12 * np.abs(want).max(), n
    assert res[widths.index(11)][0] == 5
    for i in (0, widths.index(11), widths.index(12), widths.index(13), 60, 80, 100, len(widths) - 1):
        _, one, r = solve([i])
        assert np.array_equal(one[0], xs[i], equal_nan=True) and r[0][:2] == res[i][:2], widths[i]
