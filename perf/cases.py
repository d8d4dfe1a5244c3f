"""What is timed of this framework: whole factorisations and training steps
through its public entry points, from the smallest calls to the largest.

Every case is a run of a few outer iterations from seeded initial factors, as
a user's program makes it: dense NMF (MU, HALS, ANLS-BPP), sparse NMF, NTF
(MU, HALS, ANLS-BPP) with the dimension tree, the CP loss with its gradient,
and the hierarchical rank-2 NMF.  Inputs are what these methods meet: a
non-negative low-rank model plus 1 % noise, uniform initial factors, and
power-law term-document matrices.  The one-time preparation that a program
makes once per input (the 16-bit copies, ||A||^2) is part of prepare().

The errors that a run reports are returned in FP32: they come from FP32 or
16-bit products, and their digits past that are those products' rounding.
"""
import math

import numpy as np
import torch

import planc_amd
from planc_amd import autograd

RULES = {"mu": planc_amd.MU, "hals": planc_amd.HALS, "bpp": planc_amd.ANLSBPP}
DTYPES = {"f32": planc_amd.F32, "bf16": planc_amd.BF16, "f16": planc_amd.F16}
HIER_SEED = 193957

_CTX = []


def context():
    """The one Context that a program opens and keeps."""
    if not _CTX:
        _CTX.append(planc_amd.Context(0))
    return _CTX[0]


def listed():
    return [
        # The smallest dense factorisation (the size of the smoke test): launches and latency.
        {"name": "nmf_mu_300x200", "kind": "nmf", "rule": "mu", "dtype": "f32", "m": 300, "n": 200, "k": 8, "iters": 5},
        # The first configuration of the benchmarks: a small matrix, many iterations.
        {"name": "nmf_mu_2000x1000", "kind": "nmf", "rule": "mu", "dtype": "f32", "m": 2000, "n": 1000, "k": 20,
         "iters": 20},
        # The headline: the largest dense factorisation, in mixed precision.
        {"name": "nmf_mu_65536x16384_bf16", "kind": "nmf", "rule": "mu", "dtype": "bf16", "m": 65536, "n": 16384,
         "k": 64, "iters": 10},
        # A matrix as data gives it: no dimension a multiple of anything, FP32.
        {"name": "nmf_hals_20011x9973", "kind": "nmf", "rule": "hals", "dtype": "f32", "m": 20011, "n": 9973, "k": 50,
         "iters": 5},
        # The exact alternating solver at the headline's shape: one NNLS solve per row and column.
        {"name": "nmf_bpp_65536x16384_bf16", "kind": "nmf", "rule": "bpp", "dtype": "bf16", "m": 65536, "n": 16384,
         "k": 64, "iters": 1},
        # A term-document matrix kept sparse.
        {"name": "sparse_mu_100000x40000", "kind": "sparse", "rule": "mu", "m": 100000, "n": 40000, "per_col": 80,
         "k": 32, "iters": 5},
        # The smallest tensor factorisation (the size of the smoke test).
        {"name": "ntf_hals_20x18x16", "kind": "ntf", "rule": "hals", "dtype": "f32", "dims": "20 18 16", "k": 5,
         "iters": 4},
        # A cube that fits the chip's caches: the chain of mode updates counts as much as the products.
        {"name": "ntf_hals_256c", "kind": "ntf", "rule": "hals", "dtype": "f32", "dims": "256 256 256", "k": 32,
         "iters": 9},
        # The largest tensor, in mixed precision.
        {"name": "ntf_hals_128q_f16", "kind": "ntf", "rule": "hals", "dtype": "f16", "dims": "128 128 128 128", "k": 48,
         "iters": 10},
        # A ragged four-way tensor with the exact solver.
        {"name": "ntf_bpp_61x53x47x35", "kind": "ntf", "rule": "bpp", "dtype": "f32", "dims": "61 53 47 35", "k": 17,
         "iters": 5},
        # One training step of a CP model: the loss and the gradient of every factor.
        {"name": "cp_loss_96q", "kind": "cp", "dims": "96 96 96 96", "k": 48},
        # Hierarchical topics of a term-document matrix: the complete tree.
        {"name": "hier_50000x200000", "kind": "hier", "m": 50000, "n": 200000, "per_col": 10, "depth": 9,
         "iters": 100},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["nmf", "nmf", "nmf", "sparse", "ntf", "ntf", "ntf", "cp", "hier"])
    k = _log(rng, 4, 64)
    if kind == "nmf":
        rule = rng.choice(["mu", "mu", "hals", "bpp"])
        m, n = _log(rng, 200, 65536), _log(rng, 150, 16384)
        if rng.random() < 0.4:  # sizes that a program has chosen itself
            m, n = -(-m // 16) * 16, -(-n // 16) * 16
        k = min(k, n // 10, m // 10)
        dtype = rng.choice(["f32", "f32", "bf16"] + (["f16"] if rule == "mu" else []))
        iters = rng.randint(2, 10) if rule == "mu" else rng.randint(1, 4) if rule == "hals" else 1
        iters = max(1, min(iters, int(2e10 / (m * n * (4 if dtype == "f32" else 2)))))  # no more than the headline's
        return {"kind": kind, "rule": rule, "dtype": dtype, "m": m, "n": n, "k": k, "iters": iters}
    if kind == "sparse":
        return {"kind": kind, "rule": "mu", "m": _log(rng, 2000, 100000), "n": _log(rng, 1000, 40000),
                "per_col": rng.randint(10, 80), "k": min(k, 48), "iters": rng.randint(2, 6)}
    if kind == "hier":
        return {"kind": kind, "m": _log(rng, 2000, 50000), "n": _log(rng, 5000, 200000),
                "per_col": rng.randint(6, 12), "depth": rng.randint(3, 8), "iters": rng.randint(20, 100)}
    modes = rng.choice([3, 3, 4, 4, 5])
    top = {3: 256, 4: 110, 5: 40}[modes]
    dims = [_log(rng, 12, top) for _ in range(modes)]
    if rng.random() < 0.4:
        dims = [-(-d // 4) * 4 for d in dims]
    k = min(k, 48)
    if kind == "cp":
        return {"kind": kind, "dims": " ".join(map(str, dims)), "k": k}
    rule = rng.choice(["hals", "hals", "mu", "bpp"])
    return {"kind": kind, "rule": rule, "dtype": rng.choice(["f32", "f32", "bf16", "f16"]),
            "dims": " ".join(map(str, dims)), "k": k, "iters": rng.randint(2, 12) if rule == "mu" else rng.randint(1, 4)}


def _dims(case):
    return [int(d) for d in case["dims"].split()]


# ---- inputs, from the seed alone -------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _rand(g, rows, cols):
    """U[0, 1), column-major."""
    return torch.rand((cols, rows), generator=g, device="cuda").t()


def _noise(g, like):
    """|N(0, 1)| of the shape and layout of `like`'s transpose, in slabs."""
    for i in range(0, like.shape[0], 4096):
        yield i, torch.randn((min(4096, like.shape[0] - i), like.shape[1]), generator=g, device="cuda").abs_()


def _matrix(case, seed):
    """A (m x n), and the initial W (m x k) and H (n x k)."""
    g = _gen(seed)
    m, n, k = case["m"], case["n"], case["k"]
    At = _rand(g, k, n).t().contiguous() @ _rand(g, m, k).t()  # n x m row-major: A column-major
    sigma = 0.01 * At.mean()
    for i, z in _noise(g, At):
        At[i:i + z.shape[0]].add_(z * sigma)
    return At.t(), _rand(g, m, k), _rand(g, n, k)


def _krp(factors):
    """Khatri-Rao product, the first factor's index fastest."""
    out = factors[0]
    for f in factors[1:]:
        out = (f[:, None, :] * out[None, :, :]).reshape(-1, out.shape[1])
    return out


def _tensor(case, seed):
    """X (mode 0 fastest) and the initial factors."""
    g = _gen(seed)
    dims, k = _dims(case), case["k"]
    F = [_rand(g, d, k).contiguous() for d in dims]
    s = len(dims) // 2
    X = _krp(F[s:]) @ _krp(F[:s]).t()  # (right modes) x (left modes), row-major
    sigma = 0.01 * X.mean()
    for i, z in _noise(g, X):
        X[i:i + z.shape[0]].add_(z * sigma)
    X = X.reshape(list(reversed(dims))).permute(*reversed(range(len(dims))))
    return X, [_rand(g, d, k) for d in dims]


def _documents(case, seed):
    """CSR of a term-document matrix: every document (column) draws per_col
    terms from a power law, with log-normal weights."""
    g = _gen(seed)
    m, n, per = case["m"], case["n"], case["per_col"]
    cdf = torch.cumsum(torch.arange(1, m + 1, device="cuda", dtype=torch.float64) ** -1.1, 0)
    u = torch.rand(n * per, generator=g, device="cuda", dtype=torch.float64) * cdf[-1]
    rows = torch.searchsorted(cdf, u).clamp_(max=m - 1)
    key = torch.unique(rows * n + torch.arange(n, device="cuda").repeat_interleave(per))
    data = torch.randn(key.numel(), generator=g, device="cuda").exp_()
    counts = torch.bincount(key // n, minlength=m)
    indptr = torch.zeros(m + 1, dtype=torch.int64, device="cuda")
    indptr[1:] = torch.cumsum(counts, 0)
    return indptr, (key % n).to(torch.int32), data


def _norm2(A):
    """||A||_F^2 in FP64, of a column-major matrix or a flat tensor."""
    flat = A.t() if A.dim() == 2 else A.permute(*reversed(range(A.dim())))
    return sum(float(b.double().square().sum()) for b in flat.reshape(flat.shape[0], -1).split(2048))


def prepare(case, seed):
    ctx = context()
    if case["kind"] == "nmf":
        A, W, H = _matrix(case, seed)
        s = {"A": A, "W0": W, "H0": H, "more": {"normA2": _norm2(A)}}
        if case["dtype"] != "f32":
            A16, scale = ctx.convert(A, DTYPES[case["dtype"]])
            s["more"].update(A16=A16, colscale=scale, A16T=ctx.transpose16(A16))
    elif case["kind"] == "sparse":
        g = _gen(seed + 1)
        s = {"csr": _documents(case, seed), "W0": _rand(g, case["m"], case["k"]), "H0": _rand(g, case["n"], case["k"])}
    elif case["kind"] == "ntf":
        X, F = _tensor(case, seed)
        s = {"X": X, "F0": F, "more": {"normX2": _norm2(X)}}
        if case["dtype"] != "f32":
            X16, X16T = ctx.ntf_copies16(X, DTYPES[case["dtype"]])
            s["more"].update(X16=X16, X16T=X16T)
    elif case["kind"] == "cp":
        X, F = _tensor(case, seed)
        s = {"X": X, "F0": [f.requires_grad_() for f in F]}
    else:
        indptr, indices, data = _documents(case, seed)
        s = {"csr": (indptr.cpu().numpy(), indices.cpu().numpy(), data.cpu().numpy())}
    if "W0" in s:
        s["W"], s["H"] = s["W0"].clone(), s["H0"].clone()
    elif case["kind"] == "ntf":
        s["F"] = [f.clone() for f in s["F0"]]
    s["case"] = case
    return s


def run(s):
    ctx, case = context(), s["case"]
    if case["kind"] == "nmf":
        s["W"].copy_(s["W0"])
        s["H"].copy_(s["H0"])
        rel = ctx.nmf_run(s["A"], s["W"], s["H"], RULES[case["rule"]], case["iters"], dtype=DTYPES[case["dtype"]],
                          **s["more"])
        return {"W": s["W"], "H": s["H"], "relerr": rel.astype(np.float32)}
    if case["kind"] == "sparse":
        s["W"].copy_(s["W0"])
        s["H"].copy_(s["H0"])
        rel = ctx.nmf_sparse_run(case["m"], case["n"], *s["csr"], s["W"], s["H"], RULES[case["rule"]], case["iters"])
        return {"W": s["W"], "H": s["H"], "relerr": rel.astype(np.float32)}
    if case["kind"] == "ntf":
        for f, f0 in zip(s["F"], s["F0"]):
            f.copy_(f0)
        lam, rel = ctx.ntf_run(s["X"], s["F"], RULES[case["rule"]], case["iters"], dtype=DTYPES[case["dtype"]],
                               **s["more"])
        return {"F": s["F"], "lambda": lam.float(), "relerr": rel.astype(np.float32)}
    if case["kind"] == "cp":
        loss = autograd.cp_loss(s["X"], s["F0"])
        return {"loss": loss.detach().float(), "grads": list(torch.autograd.grad(loss, s["F0"]))}
    nodes, cols, H, _ = ctx.hiernmf_run(case["m"], case["n"], *s["csr"], case["depth"], case["iters"], HIER_SEED,
                                        want_H=True)
    full = (1 << case["depth"]) - 1  # nodes too small to split leave the rest empty
    out = {"cols": cols, "H": H}
    for name, kind in (("index", np.int64), ("ncols", np.int64), ("sigma", np.float64), ("score", np.float64)):
        out[name] = np.zeros(full, dtype=kind)
        out[name][:len(nodes)] = [x[name] for x in nodes]
    return out


# ---- the work of a pass -----------------------------------------------------
def work(case):
    if case["kind"] == "hier":
        # Every level reads its entries (index and value) twice an iteration,
        # by column and by row, and both factors; the power iterations alike.
        nnz = 0.95 * case["per_col"] * case["n"]
        passes = 2 * case["depth"] * case["iters"]
        return {"bytes": passes * (16 * nnz + 16 * (case["m"] + case["n"])), "flops": passes * 8 * nnz}
    k = case["k"]
    if case["kind"] == "sparse":
        m, n, it = case["m"], case["n"], case["iters"]
        nnz = 0.8 * case["per_col"] * n
        return {"bytes": it * (2 * 8 * nnz + 4 * 4 * (m + n) * k), "flops": it * (4 * nnz * k + 4 * (m + n) * k * k)}
    if case["kind"] == "nmf":
        m, n, it = case["m"], case["n"], case["iters"]
        a = m * n * (4 if case["dtype"] == "f32" else 2)
        solve = 2.0 * (m + n) * k ** 3 / 3 if case["rule"] == "bpp" else 0  # one Cholesky per row and column
        return {"bytes": it * (2 * a + 4 * 4 * (m + n) * k),
                "flops": it * (4.0 * m * n * k + 4 * (m + n) * k * k + solve)}
    dims = _dims(case)
    numel, rows = math.prod(dims), sum(dims)
    if case["kind"] == "cp":  # the forward reads X once, the backward twice (the tree's two contractions)
        return {"bytes": 3 * 4 * numel + 2 * 4 * rows * k, "flops": 6.0 * numel * k}
    it, x = case["iters"], numel * (4 if case["dtype"] == "f32" else 2)
    solve = 2.0 * rows * k ** 3 / 3 if case["rule"] == "bpp" else 0
    return {"bytes": it * (2 * x + 3 * 4 * rows * k), "flops": it * (4.0 * numel * k + 4 * rows * k * k + solve)}


# ---- the same in 64 bits, in plain torch ------------------------------------
def _solve(T):
    """x of M x = b for a batch of [M | b], M symmetric positive definite, by
    Gauss-Jordan elimination (the library's batched Cholesky has returned
    wrong factors for large batches here)."""
    for j in range(T.shape[1]):
        row = T[:, j] / T[:, j, j, None]
        T.sub_(T[:, :, j, None] * row[:, None])
        T[:, j] = row
    return T[:, :, -1]


def _nnls(G, B):
    """argmin_x >= 0 of x^T G x / 2 - b^T x for every column b of B (k x n), by
    block principal pivoting with a backup exchange, in FP64."""
    k, n = B.shape
    X = torch.zeros_like(B)
    Y = -B
    passive = torch.zeros((n, k), dtype=torch.bool, device=B.device)
    left = torch.full((n,), k + 1, device=B.device)
    tries = torch.full((n,), 3, device=B.device)
    eye = torch.eye(k, dtype=G.dtype, device=G.device)
    order = torch.arange(k, device=B.device)
    for _ in range(5 * k):
        wrong = torch.where(passive, X.t() < 0, Y.t() < 0)
        count = wrong.sum(1)
        cols = torch.nonzero(count > 0).flatten()
        if not cols.numel():
            break
        c, w = count[cols], wrong[cols]
        better = c < left[cols]
        full = better | (tries[cols] >= 1)
        tries[cols] = torch.where(better, 3, tries[cols] - full.long())
        left[cols] = torch.where(better, c, left[cols])
        last = torch.where(w, order, -1).max(1).values
        passive[cols] ^= torch.where(full[:, None], w, order == last[:, None])
        for part in cols.split(8192):
            p = passive[part].to(G.dtype)
            M = G * p[:, :, None] * p[:, None, :] + eye * (1 - p)[:, :, None]
            rhs = (B[:, part].t() * p)[:, :, None]
            x = _solve(torch.cat([M, rhs], 2)) * p
            X[:, part] = x.t()
            Y[:, part] = G @ x.t() - B[:, part]
        X[X.abs() < 1e-12] = 0
        Y[Y.abs() < 1e-12] = 0
    return X


def _hals_rows(H, N, G):
    for x in range(H.shape[1]):
        H[:, x] = (H[:, x] + N[:, x] - H @ G[:, x]).clamp_min(1e-17)


def _normalize(W, H):
    s = W.norm(dim=0)
    W /= s
    H *= s


def _exact_nmf(rule, iters, wta, ah, norm2, W, H):
    W, H, rel = W.double().contiguous(), H.double().contiguous(), []
    if rule == "hals":
        _normalize(W, H)
    for _ in range(iters):
        if rule == "bpp":
            W = _nnls(H.t() @ H, ah(H).t().contiguous()).t().contiguous()
            N = wta(W)
            H = _nnls(W.t() @ W, N.t().contiguous()).t().contiguous()
            trace = (H * N).sum()
        else:
            N = wta(W)
            if rule == "mu":
                H = H * N / (H @ (W.t() @ W) + 1e-17)
            else:
                _hals_rows(H, N, W.t() @ W)
            N, G = ah(H), H.t() @ H
            if rule == "mu":
                W = W * N / (W @ G + 1e-17)
            else:
                for x in range(W.shape[1]):
                    w = (W[:, x] * G[x, x] + N[:, x] - W @ G[:, x]).clamp_min(1e-17)
                    W[:, x] = w / w.norm()
            trace = (W * N).sum()
        fit = norm2 - 2 * trace + ((W.t() @ W) * (H.t() @ H)).sum()
        rel.append(float((fit.clamp_min(0) / norm2).sqrt()))
        if rule == "hals":
            _normalize(W, H)
    if rule != "hals":
        _normalize(W, H)
    return {"W": _as_t(W), "H": _as_t(H), "relerr": np.array(rel)}


def _as_t(W):
    """Column-major, as the factors are stored."""
    return W.t().contiguous().t()


def _mttkrp(X, F, mode):
    """X (mode 0 fastest) times the Khatri-Rao product of the other factors (I_mode x k)."""
    dims = X.shape
    left, right = math.prod(dims[:mode]), math.prod(dims[mode + 1:])
    X2 = X.permute(*reversed(range(X.dim()))).reshape(right, dims[mode] * left)
    one = torch.ones((1, F[0].shape[1]), dtype=X.dtype, device=X.device)
    T = X2.t() @ (_krp(F[mode + 1:]) if right > 1 else one)
    return (T.reshape(dims[mode], left, -1) * (_krp(F[:mode]) if left > 1 else one)).sum(1)


def _exact_ntf(case, X, F):
    X, F, rel = X.double(), [f.double().contiguous() for f in F], []
    norm2, lam = X.square().sum(), 1.0
    for i, f in enumerate(F):
        s = f.norm(dim=0)
        F[i], lam = f / s, lam * s
    for _ in range(case["iters"]):
        for i in range(len(F)):
            S = math.prod([f.t() @ f for j, f in enumerate(F) if j != i][1:], start=(F[0] if i else F[1]).t()
                          @ (F[0] if i else F[1]))
            M = _mttkrp(X, F, i)
            if case["rule"] == "mu":
                f = F[i] * M / (F[i] @ S + 1e-6)
            elif case["rule"] == "hals":
                f = F[i].clone()
                _hals_rows(f, M, S)
            else:
                f = _nnls(S, M.t().contiguous()).t().contiguous()
            lam = f.norm(dim=0)
            F[i] = torch.where(lam > 0, f / lam, f)
        fit = norm2 - 2 * (F[-1] * lam * M).sum() + ((F[-1].t() @ F[-1]) * S * lam * lam[:, None]).sum()
        rel.append(float((fit.clamp_min(0) / norm2).sqrt()))
    return {"F": [_as_t(f) for f in F], "lambda": lam, "relerr": np.array(rel)}


def exact(case, seed):
    if case["kind"] == "nmf":
        A, W, H = _matrix(case, seed)
        A = A.double()
        return _exact_nmf(case["rule"], case["iters"], lambda f: A.t() @ f, lambda f: A @ f, A.square().sum(), W, H)
    if case["kind"] == "sparse":
        g = _gen(seed + 1)
        W, H = _rand(g, case["m"], case["k"]), _rand(g, case["n"], case["k"])
        indptr, cols, data = _documents(case, seed)
        rows = torch.repeat_interleave(torch.arange(case["m"], device="cuda"), indptr.diff())
        cols, data = cols.long(), data.double()

        def product(out, to, at):
            return lambda f: torch.zeros((out, f.shape[1]), dtype=f.dtype, device="cuda").index_add_(
                0, to, data[:, None] * f[at])
        return _exact_nmf(case["rule"], case["iters"], product(case["n"], cols, rows), product(case["m"], rows, cols),
                          data.square().sum(), W, H)
    if case["kind"] == "ntf":
        return _exact_ntf(case, *_tensor(case, seed))
    if case["kind"] == "cp":
        X, F = _tensor(case, seed)
        X, F = X.double(), [f.double() for f in F]
        s = len(F) // 2
        X2 = X.permute(*reversed(range(X.dim()))).reshape(math.prod(X.shape[s:]), -1)
        loss = 0.5 * (X2 - _krp(F[s:]) @ _krp(F[:s]).t()).square().sum()
        grads = [f @ math.prod([o.t() @ o for j, o in enumerate(F) if j != i], start=torch.ones((), device="cuda"))
                 - _mttkrp(X, F, i) for i, f in enumerate(F)]
        return {"loss": loss, "grads": [_as_t(x) for x in grads]}
    return None  # the column splits are discrete decisions of a whole tree
