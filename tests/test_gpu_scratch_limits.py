"""FP32 products where there is no room for the buffers that speed them up (the
written-out Khatri-Rao operand, the partials of K splits): the same results from
the kernels that need none.  PLANC_WS_MAX refuses buffers as a full device would.

Tolerance 3e-6, relative in the 2-norm, against FP64: FP32 accumulation of
positive terms as in the other product tests, eps * sqrt(K) for K <= 2257 in one
chain; 1e-5 for the 9000 rows of the unsplit product."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import planc_amd as P  # noqa: E402


@pytest.fixture()
def ctx():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    with P.Context(0) as c:
        yield c


def rel(x, ref):
    return np.linalg.norm(x.cpu().numpy().astype(np.float64) - ref) / np.linalg.norm(ref)


@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("dims,split,k", [((61, 13, 47), 0, 50), ((6, 10, 7, 5), 1, 8), ((5, 61, 37), 0, 17),
                                          ((41, 37, 9, 3), 1, 33)])
def test_contraction_without_room_for_its_operand(ctx, dims, split, k, side, monkeypatch):
    monkeypatch.setenv("PLANC_WS_MAX", "256")
    print("no room", dims, split, k, side, flush=True)
    rng = np.random.default_rng(sum(dims) + k)
    X = rng.random(dims).astype(np.float32)
    F = [rng.random((d, k)).astype(np.float32) for d in dims]
    out = ctx.mttkrp_partial(P.colmajor(X), [P.colmajor(f) for f in F], split, side)
    n, keep = len(dims), list(range(split + 1)) if side == 0 else list(range(split + 1, len(dims)))
    ops = [x for i in range(n) if i not in keep for x in (F[i].astype(np.float64), [i, 25])]
    ref = np.einsum(X.astype(np.float64), list(range(n)), *ops, keep + [25]).reshape((-1, k), order="F")
    assert rel(out, ref) < 3e-6


@pytest.mark.parametrize("L,K,k", [(70, 9000, 20), (1027, 515, 50)])
def test_product_without_room_for_partials(ctx, L, K, k, monkeypatch):
    monkeypatch.setenv("PLANC_WS_MAX", "256")
    print("no partials", L, K, k, flush=True)
    rng = np.random.default_rng(L)
    for ld in (L, L + 1):
        a = rng.random((L, K)).astype(np.float32)
        A = torch.as_strided(torch.zeros(ld * K, device="cuda"), (L, K), (1, ld))
        A.copy_(torch.from_numpy(a))
        b, w = rng.random((K, k)).astype(np.float32), rng.random((L, k)).astype(np.float32)
        assert rel(ctx.gemm_nn(A, P.colmajor(b)), a.astype(np.float64) @ b) < 1e-5
        assert rel(ctx.gemm_tn(A, P.colmajor(w)), w.astype(np.float64).T @ a) < 1e-5


def test_factorisation_without_room_for_the_operand(ctx, monkeypatch):
    """A whole run, its captured iterations among them: the loop's other buffers
    are there from a larger tensor whose operand needs none.  Every iteration's
    error to 1e-6 of the one with room (FP32 products of positive terms move
    err^2, here 0.2, by some 2^-24; the factors of noise move further)."""
    def run(c, dims, k, iters):
        print("ntf", dims, k, iters, flush=True)
        rng = np.random.default_rng(5)
        X = P.colmajor(rng.random(dims).astype(np.float32))
        F = [P.colmajor(rng.random((d, k)).astype(np.float32)) for d in dims]
        return c.ntf_run(X, F, P.HALS, iters)[1]

    run(ctx, (64, 64, 48, 32), 20, 12)
    with P.Context(0) as room:
        want = {n: run(room, (61, 53, 23, 31), 17, n) for n in (3, 12)}
    monkeypatch.setenv("PLANC_WS_MAX", "256")
    for n in (3, 12):
        assert np.abs(run(ctx, (61, 53, 23, 31), 17, n) - want[n]).max() < 1e-6
