"""Thin products at ragged shapes and element-aligned operands: rows that are
no multiple of 4, odd leading dimensions, bases off the 16-byte grid, and
Khatri-Rao operands with ragged factors, in every kernel family.

Against FP64 products of the same (for 16 bits: identically rounded) operands.
Tolerance, relative in the 2-norm: FP32 accumulation of K <= 700 positive
terms, eps * sqrt(K) = 3e-6, as in the aligned tests; 16 bits 1e-5."""
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


def mat(rng, rows, cols, ld, off):
    """Column-major rows x cols view with leading dimension ld, `off` elements
    into its buffer; and its values."""
    v = rng.random((rows, cols)).astype(np.float32)
    buf = torch.full((off + ld * cols,), float("nan"), dtype=torch.float32, device="cuda")
    t = torch.as_strided(buf, (rows, cols), (1, ld), off)
    t.copy_(torch.from_numpy(v))
    return t, v.astype(np.float64)


def rel(x, ref):
    return np.linalg.norm(x.cpu().numpy().astype(np.float64) - ref) / np.linalg.norm(ref)


@pytest.mark.parametrize("variant", ["", "plain", "dual", "shared"])
@pytest.mark.parametrize("L,K,k", [(3, 9, 2), (4, 16, 5), (5, 33, 17), (63, 130, 50), (65, 700, 64), (66, 129, 33),
                                   (130, 257, 16), (259, 64, 48), (1027, 515, 50)])
def test_gemm_f32_ragged(ctx, L, K, k, variant, monkeypatch):
    monkeypatch.setenv("PLANC_STREAM_VARIANT", variant)
    print("gemm ragged", L, K, k, variant, flush=True)
    rng = np.random.default_rng(L + K + k)
    for ldx, off in ((0, 0), (3, 1)):
        A, a = mat(rng, L, K, L + ldx, off)
        B, b = mat(rng, K, k, K + ldx, off)
        assert rel(ctx.gemm_nn(A, B), a @ b) < 3e-6
        B, b = mat(rng, L, k, L + ldx, off)
        assert rel(ctx.gemm_tn(A, B), b.T @ a) < 3e-6


@pytest.mark.parametrize("dt", [P.BF16, P.F16])
@pytest.mark.parametrize("L,K,k", [(5, 33, 17), (65, 700, 64), (259, 131, 48), (1027, 515, 50)])
def test_gemm_16bit_ragged(ctx, L, K, k, dt):
    print("gemm ragged 16", L, K, k, dt, flush=True)
    rng = np.random.default_rng(L + K + k)
    tt = torch.bfloat16 if dt == P.BF16 else torch.float16
    for ldx, off in ((0, 0), (3, 1)):
        v = torch.from_numpy(rng.random((L, K)).astype(np.float32)).to(tt)
        buf = torch.zeros(off + (L + ldx) * K, dtype=tt, device="cuda")
        A = torch.as_strided(buf, (L, K), (1, L + ldx), off)
        A.copy_(v)
        a, A = v.double().numpy(), A.view(torch.int16)
        for rows, product, dense in ((K, ctx.gemm_nn, lambda b: a @ b), (L, ctx.gemm_tn, lambda b: b.T @ a)):
            B, _ = mat(rng, rows, k, rows + ldx, off)
            b = B.to(tt).double().cpu().numpy()
            assert rel(product(A, B, dtype=dt), dense(b)) < 1e-5


@pytest.mark.parametrize("variant", ["", "plain", "shared", "fly"])
@pytest.mark.parametrize("dt", [P.BF16, P.F16])
@pytest.mark.parametrize("L,K,k", [(8, 33, 17), (64, 130, 50), (136, 700, 64), (1032, 515, 50), (2000, 64, 16)])
def test_gemm_16bit_nn_off_grid(ctx, L, K, k, dt, variant, monkeypatch):
    """The streaming NN kernel (rows in groups of eight) with bases and leading
    dimensions of A and B off the 16-byte grid."""
    monkeypatch.setenv("PLANC_STREAM_VARIANT", variant)
    print("gemm off grid 16", L, K, k, dt, variant, flush=True)
    rng = np.random.default_rng(L + K + k)
    tt = torch.bfloat16 if dt == P.BF16 else torch.float16
    for ldx, off in ((0, 0), (0, 1), (3, 0), (5, 3)):
        v = torch.from_numpy(rng.random((L, K)).astype(np.float32)).to(tt)
        buf = torch.zeros(off + (L + ldx) * K, dtype=tt, device="cuda")
        A = torch.as_strided(buf, (L, K), (1, L + ldx), off)
        A.copy_(v)
        B, _ = mat(rng, K, k, K + ldx, off)
        b = B.to(tt).double().cpu().numpy()
        assert rel(ctx.gemm_nn(A.view(torch.int16), B, dtype=dt), v.double().numpy() @ b) < 1e-5, (ldx, off)


@pytest.mark.parametrize("dims,k", [((7, 5, 3), 2), ((13, 9, 11), 17), ((6, 10, 7, 5), 8), ((61, 13, 47), 50)])
def test_mttkrp_ragged(ctx, dims, k):
    print("mttkrp ragged", dims, k, flush=True)
    rng = np.random.default_rng(sum(dims) + k)
    X = rng.random(dims).astype(np.float32)
    F = [rng.random((d, k)).astype(np.float32) for d in dims]
    dX, dF = P.colmajor(X), [P.colmajor(f) for f in F]
    for mode in range(len(dims)):
        sub = "abcdefg"[:len(dims)]
        ops = [x for i in range(len(dims)) if i != mode for x in (F[i].astype(np.float64), [i, 25])]
        ref = np.einsum(X.astype(np.float64), list(range(len(dims))), *ops, [25, mode])
        assert rel(ctx.mttkrp(dX, dF, mode), ref) < 3e-6, sub[mode]


def test_contraction_whose_operand_stays_unwritten(ctx):
    """Few rows against a Khatri-Rao operand of 18 MB: formed element by element."""
    dims, k = (40, 41, 43, 41), 64
    print("unwritten operand", dims, k, flush=True)
    rng = np.random.default_rng(9)
    X = rng.random(dims).astype(np.float32)
    F = [rng.random((d, k)).astype(np.float32) for d in dims]
    out = ctx.mttkrp_partial(P.colmajor(X), [P.colmajor(f) for f in F], 0, 0)
    krp = np.einsum("ax,bx,cx->cbax", *[f.astype(np.float64) for f in F[1:]]).reshape(-1, k)
    ref = X.astype(np.float64).reshape((dims[0], -1), order="F") @ krp
    assert rel(out, ref) < 3e-5  # eps * sqrt(72283)
