"""Batched BPP from the Gram and its shared inverse, against the FP64 oracle,
at the edges of its compact systems (k / 2 of 4, 8, ... 32 variables) and on
both sides of the condition limit that selects it (past it the passive systems
themselves are solved, as for up to 1024 columns of at most 16 variables).

Tolerance per column, relative to the column's largest entry: the results are
FP32 (2^-24), and the solution is refined to 1e-10 of its largest entry, so
2e-7 holds both; past the limit eps * cond is added for
the two FP64 eliminations that are compared."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import planc_amd as P  # noqa: E402
from oracle import oracle as O  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    c = P.Context(0)
    yield c
    c.close()


def problem(k, nrhs, kind):
    rng = np.random.default_rng(1000 * k + nrhs)
    A = rng.random((6 * k + 8, k))
    B = rng.random((6 * k + 8, nrhs))
    if kind == "graded":  # 1-norm condition up to a few 1e4
        A *= np.logspace(0, -1, k)
    elif kind == "ill":  # past the limit: one column nearly the sum of the others
        A[:, -1] = A[:, :-1].sum(1) / k + 1e-4 * A[:, -1]
    elif kind == "dead":  # a factor column that died: singular Gram, zero right-hand side
        A[:, k // 2] = 0.0
    return np.asfortranarray(A.T @ A), np.asfortranarray((A.T @ B).astype(np.float32))


@pytest.mark.parametrize("kind", ["plain", "graded", "ill", "dead"])
@pytest.mark.parametrize("k,nrhs", [(1, 5), (2, 70), (8, 33), (9, 64), (16, 70), (17, 1030), (31, 70), (33, 70),
                                    (48, 1030), (63, 70), (64, 1030), (1, 1030), (7, 1024), (7, 1025), (16, 3000)])
def test_bpp_pair_matches_oracle(ctx, k, nrhs, kind):
    if kind in ("ill", "dead") and k < 3:
        pytest.skip("needs other columns")
    print("bpp pair", k, nrhs, kind, flush=True)
    G, B = problem(k, nrhs, kind)
    Xr, it = O.bppnnls(G, B.astype(np.float64))
    assert it >= 0
    X = ctx.bpp(P.colmajor(G), P.colmajor(B)).cpu().numpy()
    tol = 2e-7 + (2.2e-16 * np.linalg.cond(G) if kind == "ill" else 0.0)
    err = np.abs(X - Xr).max(0) / np.maximum(np.abs(Xr).max(0), 1e-30)
    assert err.max() <= tol, (err.max(), tol)


@pytest.mark.parametrize("bad", [float("nan"), -float("inf")])
@pytest.mark.parametrize("k,nrhs", [(8, 70), (24, 70), (33, 9001), (64, 1030)])
def test_bpp_entries_that_are_no_finite_number(ctx, k, nrhs, bad):
    """A right-hand side entry of NaN or -inf is never below zero in y = G x - b,
    so its variable stays 0 and the others solve the system without it; the
    columns beside it are what they are alone.  (These columns are the ones that
    the kernel of the pair leaves to the general one, 9001 of them more than
    one pass of its grid.)"""
    print("bpp not finite", k, nrhs, bad, flush=True)
    G, B = problem(k, nrhs, "plain")
    X0 = ctx.bpp(P.colmajor(G), P.colmajor(B)).cpu().numpy()
    i, cols = k // 3, np.arange(nrhs) % 3 == 1
    Bad = B.copy(order="F")
    Bad[i, cols] = bad
    X = ctx.bpp(P.colmajor(G), P.colmajor(Bad)).cpu().numpy()
    assert np.array_equal(X[:, ~cols], X0[:, ~cols])
    rest = np.arange(k) != i
    Xr, it = O.bppnnls(np.asfortranarray(G[np.ix_(rest, rest)]), np.asfortranarray(B[np.ix_(rest, cols)].astype(np.float64)))
    assert it >= 0
    assert not X[i, cols].any()
    err = np.abs(X[np.ix_(rest, cols)] - Xr).max(0) / np.maximum(np.abs(Xr).max(0), 1e-30)
    assert err.max() <= 2e-7, err.max()
