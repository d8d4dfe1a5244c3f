"""Sparse products over rows at the edges of the row classes: empty, short,
one piece, several pieces.  FP32 sums of up to 6000 positive terms against
FP64, per element: at most as many roundings as a row has terms in one chain
(the longest is a piece's share of a lane group, 512 / 4 = 128, or a short
row's 64, plus the adding of pieces), so 160 * 2^-24 = 1e-5 relative."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import planc_amd as P  # noqa: E402
from oracle import oracle as O  # noqa: E402

LENS = [0, 1, 63, 64, 65, 0, 511, 512, 513, 1024, 1025, 6000, 3, 0]


@pytest.fixture(scope="module")
def ctx():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    c = P.Context(0)
    yield c
    c.close()


def matrix(copies=1):
    rng = np.random.default_rng(7)
    lens = LENS * copies
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    indices = np.concatenate([np.sort(rng.choice(6000, n, replace=False)) for n in lens]).astype(np.int32)
    data = (rng.random(indptr[-1]) + 0.1).astype(np.float32)
    dense = np.zeros((len(lens), 6000))
    dense[np.repeat(np.arange(len(lens)), lens), indices] = data
    return indptr, indices, data, dense


@pytest.mark.parametrize("k", [1, 3, 16, 17, 32, 33, 64])
def test_spmm_row_classes(ctx, k):
    print("spmm rows", k, flush=True)
    indptr, indices, data, dense = matrix(5)
    F = (np.random.default_rng(k).random((6000, k)) + 0.1).astype(np.float32)
    dev = [torch.from_numpy(x).cuda() for x in (indptr, indices, data)]
    out = ctx.spmm(len(dense), 6000, *dev, P.colmajor(F)).cpu().numpy()
    ref = dense @ F.astype(np.float64)
    assert np.all(out[ref == 0] == 0)
    assert np.abs(out - ref).max(initial=0, where=ref > 0) <= 1e-5 * ref.max()
    np.testing.assert_allclose(out, ref, rtol=1e-5)


@pytest.mark.parametrize("k", [3, 17, 40])
def test_nmf_sparse_row_classes(ctx, k):
    """One MU iteration (products by rows and, transposed, by columns)."""
    print("sparse nmf rows", k, flush=True)
    indptr, indices, data, dense = matrix(4)
    m, n = dense.shape
    rng = np.random.default_rng(k)
    W0, H0 = (rng.random((d, k)).astype(np.float32) for d in (m, n))
    Wr, Hr, rel, rc = O.nmf_sparse(P.MU, m, n, indptr, indices, data.astype(np.float64), W0.astype(np.float64),
                                   H0.astype(np.float64), 1)
    assert rc == 0
    dW, dH = P.colmajor(W0), P.colmajor(H0)
    got = ctx.nmf_sparse_run(m, n, *[torch.from_numpy(x).cuda() for x in (indptr, indices, data)], dW, dH, P.MU, 1)
    assert abs(got[0] - rel[0]) < 1e-6
    for x, r in ((dW, Wr), (dH, Hr)):
        assert np.linalg.norm(x.cpu().numpy() - r) < 1e-5 * np.linalg.norm(r)


def elapsed(f, reps):
    """Microseconds per call, the best of three runs after one call."""
    f()
    best = float("inf")
    for _ in range(3):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for _ in range(reps):
            f()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) * 1000 / reps)
    return best


@pytest.mark.parametrize("k", [8, 16])
def test_spmm_long_rows_run_side_by_side(ctx, k):
    """Rows just past the short class take no more than twice the time of rows
    just inside it (10000 rows of 66 and of 64 entries): a wavefront each, not one
    after the other in a block."""
    g = torch.Generator(device="cuda").manual_seed(k)
    F = torch.rand((k, 5000), generator=g, device="cuda").t()

    def run(per):
        print("spmm rows of", per, k, flush=True)
        indptr = torch.arange(10001, device="cuda", dtype=torch.int64) * per
        idx = torch.randint(0, 5000, (10000 * per,), generator=g, device="cuda", dtype=torch.int32)
        val = torch.rand(10000 * per, generator=g, device="cuda")
        return elapsed(lambda: ctx.spmm(10000, 5000, indptr, idx, val, F), 50)

    short, long = run(64), run(66)
    assert long <= 2 * short, (short, long)


@pytest.mark.parametrize("where", ["first", "last", "spread", "none"])
def test_transpose_with_empty_columns(ctx, where):
    """Row pointers of the transpose over long runs of empty columns: right, and
    in time that does not grow with a run's length (20000 columns a millisecond
    would be one lane writing them one by one)."""
    print("transpose", where, flush=True)
    m, n = 1000, 2_000_000
    per = 0 if where == "none" else 3
    rng = np.random.default_rng(1)
    if where == "spread":
        cols = np.sort(np.stack([rng.choice(n, 3, replace=False) for _ in range(m)]), axis=1)
    else:
        cols = np.sort(np.stack([rng.choice(50, 3, replace=False) for _ in range(m)]), axis=1) + (n - 50) * (where == "last")
    cols = cols[:, :per].reshape(-1).astype(np.int32)
    data = rng.random(m * per).astype(np.float32)
    indptr = (np.arange(m + 1) * per).astype(np.int64)
    dev = [torch.from_numpy(x).cuda() for x in (indptr, cols, data)]
    if not per:
        dev[1:] = [torch.empty(0, dtype=t, device="cuda") for t in (torch.int32, torch.float32)]
    tp, ti, tv = (x.cpu().numpy() for x in ctx.csr_transpose(m, n, *dev))
    order = np.argsort(cols, kind="stable")
    assert np.array_equal(tp, np.concatenate([[0], np.cumsum(np.bincount(cols, minlength=n))]))
    assert np.array_equal(ti, np.repeat(np.arange(m), per)[order])
    assert np.array_equal(tv, data[order])
    assert elapsed(lambda: ctx.csr_transpose(m, n, *dev), 3) < 10000
