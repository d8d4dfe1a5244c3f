"""NMF errors of several iterations formed by one launch, against the residual of
the factors: runs that end at the first, a middle and the last place of a batch
report ||A - W H^T|| / ||A|| of what they return, and a longer run the same on its
way.

The reported error is a difference of sums, err^2 = (||A||^2 - 2 <W, A H> +
<W^T W, H^T H>) / ||A||^2, of which <W, A H> comes from FP32 products: their
roundings, 2^-24 times some 8 per element and averaged over 1500 elements and
more, leave 1e-8 of err^2, and err is 0.01 and up: 1e-6.  Two runs of the same
loop agree to their FP64 sums, 1e-10.  Early errors differ by 1e-4 and more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import planc_amd as P  # noqa: E402
from planc_amd import datagen as D  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    c = P.Context(0)
    yield c
    c.close()


# The first shape's rows and Grams are updated in one pass, the second's apart.
@pytest.mark.parametrize("m,n,k", [(300, 200, 8), (1501, 333, 20)])
@pytest.mark.parametrize("algo", [P.MU, P.HALS, P.ANLSBPP])
def test_errors_are_the_residuals(ctx, algo, m, n, k):
    a = D.lowrank_matrix(m, n, k, 0.05, stream=3).astype(np.float32)
    A, a = P.colmajor(a), a.astype(np.float64)
    W0, H0 = D.init_factors([(m, k), (n, k)], stream=4)

    def run(iters):
        print(f"algo={algo} {m}x{n} k={k} iters={iters}", flush=True)
        W, H = P.colmajor(W0.astype(np.float32)), P.colmajor(H0.astype(np.float32))
        rel = np.asarray(ctx.nmf_run(A, W, H, algo, iters))
        assert rel.shape == (iters,)
        w, h = (x.cpu().numpy().astype(np.float64) for x in (W, H))
        return rel, np.linalg.norm(a - w @ h.T) / np.linalg.norm(a)

    full, _ = run(40)
    if algo != P.ANLSBPP:
        assert full[0] - full[1] > 1e-4
    for iters in (1, 2, 3, 15, 16, 17, 18, 31, 32, 33, 40):
        rel, residual = run(iters)
        if algo != P.ANLSBPP:  # whose errors are formed one by one
            assert abs(rel[-1] - residual) <= 1e-6, iters
        assert np.abs(rel - full[:iters]).max() <= 1e-10
