"""Timed cases of the QR library's public entry points, from a single small
panel to the 32768×4096 factorization.

A case is a dict of plain values; `kind` names the entry point:
  panel  hh_recon_qr: TSQR + Householder reconstruction of one m×b panel
  qr2d   QR_2D: blocked QR of an m×n matrix with panels of width b
  lstsq  lstsq: factorization, solve and FP64 refinement
  batch  Batch.qr: many independent tall-skinny factorizations at once
  served lstsq_batched: many small least-squares requests at once
  apply  apply_tsqr_QT: the implicit TSQR Q (or Qᵀ) applied to m×k columns

The library factors in place, so a pass that factors starts with a device
copy of the matrix its caller keeps.  Matrices are flat column-major.
"""
import numpy as np
import torch

from candmc_amd import qr

DEV = "cuda:0"
F64 = torch.float64


def listed():
    return [
        # the smallest panel: one leaf, all latency and launches
        dict(name="panel_256x16", kind="panel", m=256, b=16, ranks=0, factors=False),
        # the reference test's panel over four ranks, with T and T⁻ᵀ as upd_A takes them
        dict(name="panel_8192x64_r4", kind="panel", m=8192, b=64, ranks=4, factors=True),
        # one full-height panel of the large factorization
        dict(name="panel_32768x128", kind="panel", m=32768, b=128, ranks=0, factors=True),
        # odd rows and a width that is no multiple of a tile
        dict(name="panel_4099x100", kind="panel", m=4099, b=100, ranks=0, factors=False),
        # the smallest blocked factorization: a chain of short launches
        dict(name="qr2d_160x96_b32", kind="qr2d", m=160, n=96, b=32),
        # an ordinary ragged matrix (odd leading dimension, a partial last panel)
        dict(name="qr2d_8193x1500_b128", kind="qr2d", m=8193, n=1500, b=128),
        # the large factorization of the benchmark
        dict(name="qr2d_32768x4096_b128", kind="qr2d", m=32768, n=4096, b=128),
        # least squares: the large FP64 solve, and a ragged one with the FP32 update
        dict(name="lstsq_65536x2048_f64", kind="lstsq", m=65536, n=2048, nrhs=1, prec="f64", kappa=1e6),
        dict(name="lstsq_16500x1100_f32", kind="lstsq", m=16500, n=1100, nrhs=5, prec="f32", kappa=1e2),
        # a batch of tall-skinny problems of uneven sizes, m in [256, 16384], n in {16, 32, 64, 128}
        dict(name="batch_512", kind="batch", nprob=512, sizes=13, dtype="f64"),
        # a server's batch of queued one-panel requests of one width
        dict(name="served_32x64", kind="served", nprob=32, n=64, sizes=17, kappa=1e3),
        # the implicit Qᵀ of a panel's tree on trailing columns
        dict(name="apply_qt_32768x128_k2000", kind="apply", m=32768, b=128, ranks=128, k=2000, trans=True),
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], spread evenly over its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["panel", "panel", "qr2d", "qr2d", "qr2d", "lstsq", "batch", "served", "apply"])
    if kind == "panel":
        b = rng.choice([16, 32, 64, 100, 128, rng.randint(8, 128)])
        m = _log(rng, max(256, b), 65536)
        return dict(kind=kind, m=m, b=b, ranks=rng.choice([0, 0, 4]) if m >= 8 * b else 0, factors=rng.random() < 0.5)
    if kind == "qr2d":
        m = _log(rng, 160, 32768)
        n = _log(rng, 48, min(4096, 3 * m // 4))
        return dict(kind=kind, m=m, n=n, b=rng.choice([32, 64, 96, 128, 128, 128]) if n < 1500 else 128)
    if kind == "lstsq":
        m = _log(rng, 1024, 65536)
        n = _log(rng, 64, min(2048, m // 4))
        f32 = rng.random() < 0.4
        return dict(kind=kind, m=m, n=n, nrhs=rng.randint(1, 16), prec="f32" if f32 else "f64",
                    kappa=1e2 if f32 else 10.0 ** rng.randint(1, 6))
    if kind == "batch":
        return dict(kind=kind, nprob=_log(rng, 16, 512), sizes=rng.randint(1, 1 << 30),
                    dtype=rng.choice(["f64", "f64", "f32"]))
    if kind == "served":
        return dict(kind=kind, nprob=_log(rng, 2, 32), n=rng.randint(8, 128), sizes=rng.randint(1, 1 << 30),
                    kappa=10.0 ** rng.randint(0, 6))
    b = rng.choice([32, 64, 128])
    ranks = _log(rng, 4, 128)
    return dict(kind=kind, m=ranks * rng.randint(b, 256), b=b, ranks=ranks, k=_log(rng, 100, 2000),
                trans=rng.random() < 0.5)


# --- inputs -------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(gen, count):
    return torch.randn(count, generator=gen, dtype=F64, device=DEV)


def _scaled(gen, m, n, kappa):
    """m×n N(0,1) entries, columns scaled geometrically from 1 to 1/kappa (flat column-major)."""
    s = torch.logspace(0, -float(np.log10(kappa)), n, dtype=F64, device=DEV)
    return (_randn(gen, m * n).reshape(n, m) * s[:, None]).reshape(-1)


def _batch_sizes(case):
    r = np.random.default_rng(case["sizes"])
    return r.integers(256, 16385, case["nprob"]), r.choice([16, 32, 64, 128], case["nprob"])


def _served_sizes(case):
    """Rows lognormal around 4096, 1 to 16 right-hand sides, as a request stream has them."""
    r = np.random.default_rng(case["sizes"])
    m = np.clip(r.lognormal(np.log(4096), 1.0, case["nprob"]), case["n"], 65536).astype(np.int64)
    return m, r.integers(1, 17, case["nprob"])


def _inputs(case, seed):
    """The random inputs alone (what `prepare` and `exact` share)."""
    g, kind = _gen(seed), case["kind"]
    if kind == "panel":
        return _randn(g, case["m"] * case["b"])
    if kind == "qr2d":
        return _randn(g, case["m"] * case["n"])
    if kind == "lstsq":
        return _scaled(g, case["m"], case["n"], case["kappa"]), _randn(g, case["m"] * case["nrhs"])
    if kind == "batch":
        m, n = _batch_sizes(case)
        A = _randn(g, int(np.sum(m * n)))
        return A.float() if case["dtype"] == "f32" else A
    if kind == "served":
        m, k = _served_sizes(case)
        return [(_scaled(g, int(mp), case["n"], case["kappa"]), _randn(g, int(mp * kp))) for mp, kp in zip(m, k)]
    return _randn(g, case["m"] * case["b"]), _randn(g, case["m"] * case["k"])


def prepare(case, seed):
    kind = case["kind"]
    inp = _inputs(case, seed)
    st = dict(case=case, inp=inp)
    if kind == "panel":
        bb = case["b"] * case["b"]
        st["A"] = torch.empty_like(inp)
        st["W"] = torch.zeros(bb, dtype=F64, device=DEV)
        st["T"] = torch.zeros(bb, dtype=F64, device=DEV) if case["factors"] else None
        st["Ti"] = torch.zeros(bb, dtype=F64, device=DEV) if case["factors"] else None
    elif kind == "qr2d":
        st["A"] = torch.empty_like(inp)
    elif kind == "lstsq":
        st["X"] = torch.zeros(case["n"] * case["nrhs"], dtype=F64, device=DEV)
    elif kind == "batch":
        m, n = _batch_sizes(case)
        st["plan"] = qr.Batch(m, n)
        st["A"] = torch.empty_like(inp)
        st["Tt"] = st["plan"].new_t(inp)
    elif kind == "served":
        n = case["n"]
        m, k = _served_sizes(case)
        st["X"] = [torch.zeros(n * int(kp), dtype=F64, device=DEV) for kp in k]
        st["reqs"] = [(A, int(mp), int(mp), n, B, int(mp), int(kp), X, n)
                      for (A, B), X, mp, kp in zip(inp, st["X"], m, k)]
    else:
        m, b, P = case["m"], case["b"], case["ranks"]
        st["Y"] = inp[0].clone()
        st["tau"] = torch.zeros(P * b, dtype=F64, device=DEV)
        st["td"] = torch.zeros(qr.tree_data_size(m, b, P), dtype=F64, device=DEV)
        R = torch.zeros(b * b, dtype=F64, device=DEV)
        qr.bitree_tsqr(st["Y"], m, R, st["tau"], m, b, numPes=P, output_Y=1, tree_data=st["td"])
        st["B"] = torch.empty_like(inp[1])
    return st


def run(st):
    case, kind = st["case"], st["case"]["kind"]
    if kind == "panel":
        st["A"].copy_(st["inp"])
        qr.hh_recon_qr(st["A"], case["m"], case["m"], case["b"], st["W"], numPes=case["ranks"], T=st["T"],
                       invT_T=st["Ti"], sync=False)
        return [x for x in (st["A"], st["W"], st["T"], st["Ti"]) if x is not None]
    if kind == "qr2d":
        st["A"].copy_(st["inp"])
        qr.QR_2D(st["A"], case["m"], case["m"], case["n"], case["b"], sync=False)
        return st["A"]
    if kind == "lstsq":
        A, B = st["inp"]
        m, n, f32 = case["m"], case["n"], case["prec"] == "f32"
        X, _, _ = qr.lstsq(A, m, m, n, B, m, case["nrhs"], X=st["X"], prec=qr.PREC_F32 if f32 else qr.PREC_F64,
                           max_iter=10, tol=1e-10 if f32 else 1e-12)
        return X
    if kind == "batch":
        st["A"].copy_(st["inp"])
        st["plan"].qr(st["A"], st["Tt"], sync=False)
        return [st["A"], st["Tt"]]
    if kind == "served":
        qr.lstsq_batched(st["reqs"])
        return list(st["X"])
    m, b, k = case["m"], case["b"], case["k"]
    st["B"].copy_(st["inp"][1])
    qr.apply_tsqr_QT(st["Y"], m, st["tau"], st["B"], m, m, b, k, numPes=case["ranks"], tree_data=st["td"],
                     trans=case["trans"], sync=False)
    return st["B"]


# --- what a pass cannot do without ----------------------------------------------
def _qr_flops(m, n):
    return 2.0 * m * n * n - 2.0 / 3.0 * n ** 3


def work(case):
    kind = case["kind"]
    if kind in ("panel", "qr2d"):
        m, n = case["m"], case["b"] if kind == "panel" else case["n"]
        return {"bytes": 16 * m * n, "flops": int(_qr_flops(m, n))}
    if kind == "lstsq":
        m, n, k = case["m"], case["n"], case["nrhs"]
        return {"bytes": 8 * (m * n + m * k + n * k), "flops": int(_qr_flops(m, n) + 4.0 * m * n * k)}
    if kind == "batch":
        m, n = (x.astype(np.float64) for x in _batch_sizes(case))
        size = 4 if case["dtype"] == "f32" else 8
        return {"bytes": int(np.sum(2 * size * m * n + size * n * n)), "flops": int(np.sum(_qr_flops(m, n)))}
    if kind == "served":
        n = float(case["n"])
        m, k = (x.astype(np.float64) for x in _served_sizes(case))
        return {"bytes": int(np.sum(8 * (m * n + m * k + n * k))), "flops": int(np.sum(_qr_flops(m, n) + 4 * m * n * k))}
    m, b, k = case["m"], case["b"], case["k"]
    return {"bytes": 8 * (m * b + 2 * m * k), "flops": int(4.0 * m * b * k)}


# --- the same results from LAPACK ------------------------------------------------
def _dense(flat, m, n):
    """Host m×n matrix of a flat column-major tensor, FP64."""
    return flat.to(device="cpu", dtype=F64).reshape(n, m).T


def _flat(M):
    return M.T.contiguous().reshape(-1)


def _panel_factors(A):
    """[Y\\R], W, T and T⁻ᵀ of Q = I − Y·T·Yᵀ from dgeqrf: T⁻¹ = striu(YᵀY) + diag(YᵀY)/2 and
    W = −T·Y1ᵀ; a reflector with tau = 0 (a last row's) makes its row and column of T zero."""
    b = A.shape[1]
    YR, tau = torch.geqrf(A)
    Y = torch.tril(YR, -1)
    Y[range(b), range(b)] = 1.0
    G = Y.T @ Y
    T = torch.zeros(b, b, dtype=F64)
    for i in range(b):
        T[:i, i] = -tau[i] * (T[:i, :i] @ G[:i, i])
        T[i, i] = tau[i]
    Ti = torch.tril(G)
    Ti[range(b), range(b)] *= 0.5
    return YR, -T @ Y[:b].T, T, Ti


def _apply_tree(A, B, m, b, P, trans):
    """Q or Qᵀ of the binary tree over P equal row blocks: dgeqrf of each block, then receiver z
    stacked on sender z + ceil(n/2) on each level of n live ranks."""
    off = [(p * m) // P for p in range(P + 1)]
    B = B.clone()
    leaf, R = [], []
    for p in range(P):
        a, tau = torch.geqrf(A[off[p]:off[p + 1]])
        leaf.append((a, tau))
        R.append(torch.triu(a[:b]))
    nodes, n = [], P
    while n > 1:
        half = (n + 1) // 2
        for z in range(n // 2):
            a, tau = torch.geqrf(torch.cat([R[z], R[z + half]]))
            nodes.append((z, z + half, a, tau))
            R[z] = torch.triu(a[:b])
        n = half

    def leaves():
        for p in range(P):
            B[off[p]:off[p + 1]] = torch.ormqr(*leaf[p], B[off[p]:off[p + 1]], left=True, transpose=trans)

    def tree(order):
        for z, s, a, tau in order:
            x = torch.cat([B[off[z]:off[z] + b], B[off[s]:off[s] + b]])
            x = torch.ormqr(a, tau, x, left=True, transpose=trans)
            B[off[z]:off[z] + b], B[off[s]:off[s] + b] = x[:b], x[b:]

    if trans:
        leaves()
        tree(nodes)
    else:
        tree(nodes[::-1])
        leaves()
    return B


def exact(case, seed):
    kind = case["kind"]
    inp = _inputs(case, seed)
    if kind == "panel":
        out = _panel_factors(_dense(inp, case["m"], case["b"]))
        return [_flat(x) for x in (out if case["factors"] else out[:2])]
    if kind == "qr2d":
        return _flat(torch.geqrf(_dense(inp, case["m"], case["n"]))[0])
    if kind in ("lstsq", "served"):
        def solve(A, B, m, n, k):
            return _flat(torch.linalg.lstsq(_dense(A, m, n), _dense(B, m, k), driver="gels").solution[:n])
        if kind == "lstsq":
            return solve(*inp, case["m"], case["n"], case["nrhs"])
        m, k = _served_sizes(case)
        return [solve(A, B, int(mp), case["n"], int(kp)) for (A, B), mp, kp in zip(inp, m, k)]
    if kind == "batch":
        m, n = _batch_sizes(case)
        A, Tt, at = torch.empty(inp.numel(), dtype=F64), [], 0
        host = inp.to(device="cpu", dtype=F64)
        for mp, np_ in zip(m.tolist(), n.tolist()):
            YR, _, T, _ = _panel_factors(host[at:at + mp * np_].reshape(np_, mp).T)
            A[at:at + mp * np_] = _flat(YR)
            Tt.append(T.contiguous().reshape(-1))      # Tᵀ, column-major
            at += mp * np_
        return [A, torch.cat(Tt)]
    m, b, k = case["m"], case["b"], case["k"]
    return _flat(_apply_tree(_dense(inp[0], m, b), _dense(inp[1], m, k), m, b, case["ranks"], case["trans"]))
