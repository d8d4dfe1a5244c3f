"""The first call of a shape, which chooses its products' kernels by timing them,
against the calls after it.  For a matrix or tensor of a few MB the choice may
cost a few calls, not tens (a first call of five NMF-MU iterations on 2000 x 1000
took 2.8 calls when this was written, of NTF-HALS 61 x 53 x 47 x 35 2.1; with every
split count among the candidates 11 and 16)."""
import time

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import planc_amd as P  # noqa: E402


def rand(g, rows, cols):
    return torch.rand((cols, rows), generator=g, device="cuda").t()


def first_and_later(make):
    """Seconds of the first call in a new context (the best of three contexts,
    after one that loads the kernels) and of the best of eight more."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    first, later = [], []
    for i in range(4):
        with P.Context(0) as c:
            call = make(c)
            for j in range(9):
                torch.cuda.synchronize()
                t = time.perf_counter()
                call()
                torch.cuda.synchronize()
                if i:
                    (later if j else first).append(time.perf_counter() - t)
    return min(first), min(later)


@pytest.mark.parametrize("m,n,k", [(2000, 1000, 20), (400, 16384, 16)])
def test_nmf(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(1)
    A, W, H = rand(g, m, n), rand(g, m, k), rand(g, n, k)
    first, later = first_and_later(lambda c: lambda: c.nmf_run(A, W.clone(), H.clone(), P.MU, 5))
    print("nmf", m, n, k, first, later, flush=True)
    assert first < 6 * later


def test_ntf():
    g = torch.Generator(device="cuda").manual_seed(1)
    dims, k = (61, 53, 47, 35), 17
    X = torch.rand(tuple(reversed(dims)), generator=g, device="cuda").permute(3, 2, 1, 0)
    F = [rand(g, d, k) for d in dims]
    first, later = first_and_later(lambda c: lambda: c.ntf_run(X, [f.clone() for f in F], P.HALS, 3))
    print("ntf", dims, k, first, later, flush=True)
    assert first < 6 * later
