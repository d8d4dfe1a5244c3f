"""How the sums of FP32 products are cut into accumulator chains: a tensor
contraction over at most 320 rows and any product over at most 128 not at all, a
product of an operand off the 16-byte grid into at most 1024 rows.

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
    ((12, 320), 0, 5),         # the limit itself
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


def chain_loss(c, trans, L, K, ld, off):
    """Least number of the K - 1 ones that a product keeps beside a first row of
    2^27.  Chains but the first one's add whole (multiples of 16 rows, but the
    last one's rest)."""
    rows, cols = (K, L) if trans else (L, K)
    ldr = -(-rows // 4) * 4 + ld
    buf = torch.ones(off + ldr * cols, device="cuda")
    A = torch.as_strided(buf, (rows, cols), (1, ldr), off)
    if trans:
        A[0, :] = 2.0 ** 27
    else:
        A[:, 0] = 2.0 ** 27
    B = torch.ones((5, K), device="cuda").t()
    out = (c.gemm_tn if trans else c.gemm_nn)(A, B)
    return (out.double() - 2.0 ** 27).min().item()


@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("L,K", [(60, 50), (3000, 100), (5, 33), (200, 128)])
def test_short_products_are_not_split(trans, L, K):
    print("short product", trans, L, K, flush=True)
    with P.Context(0) as c:
        assert chain_loss(c, trans, L, K, 0, 0) == 0


@pytest.mark.parametrize("tune", ["0", "1"])
@pytest.mark.parametrize("ld,off", [(3, 0), (0, 1), (1, 2)])
@pytest.mark.parametrize("trans,L,K", [(0, 16400, 6000), (1, 16400, 6000), (0, 70, 9000), (1, 40, 9000),
                                       (0, 70001, 20001)])
def test_chains_of_1024_rows_at_most(trans, L, K, ld, off, tune, monkeypatch):
    """Operands off the 16-byte grid: an accumulator takes at most 1024 rows, so
    the first row's term swallows no more than those ones."""
    monkeypatch.setenv("PLANC_AUTOTUNE", tune)
    print("chain limit", trans, L, K, ld, off, tune, flush=True)
    with P.Context(0) as c:  # the choice of another test's timings is not this one's
        assert chain_loss(c, trans, L, K, ld, off) >= K - 1 - 1024 - 64


@pytest.mark.parametrize("trans", [0, 1])
def test_chain_limit_after_an_aligned_call(trans, monkeypatch):
    """The same shape and leading dimension on the grid first, whose choice is
    its own."""
    monkeypatch.setenv("PLANC_AUTOTUNE", "0")
    print("chain limit after an aligned call", trans, flush=True)
    with P.Context(0) as c:
        chain_loss(c, trans, 16400, 6000, 0, 0)
        assert chain_loss(c, trans, 16400, 6000, 0, 1) >= 6000 - 1 - 1024 - 64
