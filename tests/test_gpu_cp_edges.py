"""CP loss and gradient where the fused forward's tiles end: extents around the
16-byte loads, the 64-row and 128-column tiles and the 16-column rank steps.

Loss: an FP32 model value of k terms against X leaves residuals good to about
k * 6e-8 of X; relative to a loss of random X (residual of X's own size) that is
64 * 6e-8 = 4e-6 and averages out over the entries: 1e-5.  Gradient: FP32 products
over at most 7000 entries, 6e-8 * sqrt(7000) = 5e-6 of a sum that cancels by less
than a factor 10: 1e-4.
"""
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


@pytest.mark.parametrize("dims,k", [((1, 1), 1), ((63, 127), 16), ((64, 128), 17), ((65, 129), 33), ((66, 130), 64),
                                    ((3, 5, 7), 1), ((67, 2, 65), 15), ((4, 16, 32), 49), ((68, 1, 131), 32),
                                    ((13, 5, 11, 9), 48), ((3, 2, 5, 2, 7), 20), ((2, 3, 2, 3, 2, 3), 5)])
def test_cp_loss_edges(ctx, dims, k):
    print(f"cp edges {dims} k={k}", flush=True)
    rng = np.random.default_rng(sum(dims) + k)
    X = np.asfortranarray(rng.random(dims, dtype=np.float32) * k)
    F = [rng.random((d, k), dtype=np.float32) for d in dims]
    ref, gref = O.cp_loss(X.astype(np.float64), [f.astype(np.float64) for f in F], grads=True)
    dX, dF = P.colmajor(X), [P.colmajor(f) for f in F]
    assert abs(ctx.cp_loss(dX, dF) - ref) <= 1e-5 * ref
    if len(dims) < 3:  # the gradient takes three modes and more
        return
    for g, r in zip(ctx.cp_loss_grad(dX, dF), gref):
        assert np.linalg.norm(g.cpu().numpy() - r) <= 1e-4 * np.linalg.norm(r)
