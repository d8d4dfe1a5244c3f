"""NMF errors of several iterations formed by one launch: iteration counts on
both sides of a full batch give the errors that the iterations have one by one.

A loop of n iterations does what the first n of a longer loop do, so the errors
agree to the rounding of their FP64 sums: 1e-16 times some 50 for the sums'
length, over the squared error (7e-5 and up) that the subtraction leaves: 1e-10.
"""
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


@pytest.mark.parametrize("m,n,k", [(300, 200, 7), (1501, 333, 20)])
@pytest.mark.parametrize("algo", [P.MU, P.HALS, P.ANLSBPP])
def test_errors_do_not_depend_on_the_batch(ctx, algo, m, n, k):
    A = P.colmajor(D.lowrank_matrix(m, n, k, 0.05, stream=3).astype(np.float32))
    W0, H0 = D.init_factors([(m, k), (n, k)], stream=4)

    def run(iters):
        print(f"algo={algo} {m}x{n} k={k} iters={iters}", flush=True)
        W, H = P.colmajor(W0.astype(np.float32)), P.colmajor(H0.astype(np.float32))
        return np.asarray(ctx.nmf_run(A, W, H, algo, iters))

    full = run(33)
    assert full.shape == (33,)
    for iters in (1, 15, 16, 17, 32):
        rel = run(iters)
        assert rel.shape == (iters,)
        assert np.abs(rel - full[:iters]).max() <= 1e-10
