"""FP32 tensor contractions over at most 512 rows are summed in one chain.

The first term of every sum is 2^27 and the others are ones: an FP32
accumulator that holds 2^27 (unit in the last place 16) takes a matrix step's
four of them without a change, so one chain over all rows gives 2^27 exactly.  A
sum that is cut into pieces of 16 rows or more adds each further piece whole."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import planc_amd as P  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    c = P.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("dims,split,k", [
    ((20, 18, 16), 0, 5),      # ragged first right factor: the operand is written out
    ((20, 16, 16), 0, 5),      # formed in the kernel
    ((288, 20, 3), 0, 17),     # one left factor
    ((16, 18, 20, 2), 1, 33),  # a ragged pair on the left
    ((12, 512), 0, 5),         # the limit itself
])
def test_one_chain(ctx, dims, split, k, side):
    print("one chain", dims, split, k, side, flush=True)
    L = int(np.prod(dims[:split + 1]))
    R = int(np.prod(dims[split + 1:]))
    X = np.ones((L, R), dtype=np.float32)
    if side == 0:
        X[:, 0] = 2.0 ** 27
    else:
        X[0, :] = 2.0 ** 27
    dX = P.colmajor(X.reshape(dims, order="F"))
    F = [P.colmajor(np.ones((d, k), dtype=np.float32)) for d in dims]
    out = ctx.mttkrp_partial(dX, F, split, side).cpu().numpy()
    assert np.array_equal(out, np.full(out.shape, 2.0 ** 27, dtype=np.float32))
