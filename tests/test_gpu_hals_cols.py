"""HALS column sweep at the edges of its layout: ranks around each register
width and around the groups of four columns, row counts around each block size
and past the widest blocks' launch, against the same sweep in FP64.

Tolerance 1e-4 of the factor's norm: a row's dot has up to 64 terms of size
about 10 (G of 40 rows in [0, 1]), summed in FP32 (6e-8), against values of
order 1 that remain after the subtraction: 64 * 10 * 6e-8 = 4e-5.
"""
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


@pytest.mark.parametrize("m,k", [(1, 1), (7, 3), (255, 4), (1025, 5), (1024, 15), (513, 16), (2047, 17), (511, 31),
                                 (4097, 32), (513, 33), (20011, 48), (512, 49), (1023, 61), (20011, 64),
                                 (140000, 40), (140000, 52), (300000, 20)])
def test_sweep_edges(ctx, m, k):
    print(f"hals cols m={m} k={k}", flush=True)
    rng = np.random.default_rng(m + 100 * k)
    W = rng.random((m, k), dtype=np.float32)
    AH = rng.random((m, k), dtype=np.float32) * 5
    Ht = rng.random((40, k))
    G = Ht.T @ Ht
    dW = P.colmajor(W)
    ctx.hals_update_cols(dW, P.colmajor(AH), P.colmajor(G))
    ref = W.astype(np.float64)
    for x in range(k):
        v = ref[:, x] * G[x, x] + (AH[:, x].astype(np.float64) - ref @ G[:, x])
        v = np.where(v < 1e-17, 1e-17, v)
        ref[:, x] = v / np.linalg.norm(v)
    got = dW.cpu().numpy().astype(np.float64)
    assert np.linalg.norm(got - ref) <= 1e-4 * np.linalg.norm(ref)
