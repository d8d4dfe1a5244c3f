"""Hierarchical rank-2 tree with rows on both sides of each length class (8, 128,
1024 and 4096 entries) against the oracle's node-by-node tree.  Same FP64
arithmetic in another order: 1e-9, as for the other trees."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import planc_amd as P  # noqa: E402
from test_gpu_parity import _hier_reference, rel_err  # noqa: E402


@pytest.mark.parametrize("lens", [[1, 2, 7, 8, 9, 10, 15, 16, 17, 3, 5, 6], [127, 128, 129, 8, 64, 65, 120, 40],
                                  [1023, 1024, 1025, 130, 9, 30, 4, 511], [4095, 4096, 4097, 129, 12, 8193, 77, 20]])
def test_row_classes(lens):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    print(f"hier rows {lens}", flush=True)
    n, depth, iters, seed = 9000 if max(lens) > 200 else 300, 3, 8, 77
    rng = np.random.default_rng(sum(lens))
    lens = np.array(lens * 20 if max(lens) < 200 else lens + [25] * 150)
    m = len(lens)
    ix = np.concatenate([np.sort(rng.choice(n, size=int(c), replace=False)) for c in lens]).astype(np.int32)
    ip = np.zeros(m + 1, dtype=np.int64)
    ip[1:] = np.cumsum(lens)
    dv = rng.lognormal(0.0, 1.0, size=int(ip[-1])).astype(np.float32)
    ref = _hier_reference(m, n, ip, ix, dv.astype(np.float64), depth, iters, seed)
    ctx = P.Context(0)
    out, cols, H, W = ctx.hiernmf_run(m, n, ip, ix, dv, depth, iters, seed, want_H=True, want_W=True)
    ctx.close()
    assert len(out) == len(ref)
    for o, r in zip(out, ref):
        assert o["index"] == r["index"] and o["level"] == r["level"]
        assert np.array_equal(cols[o["col_offset"]:o["col_offset"] + o["ncols"]], r["cols"])
        if r["level"] > 0:
            assert abs(o["sigma"] - r["sigma"]) <= 1e-9 * max(1.0, r["sigma"])
        if "H" in r:
            h = H[2 * o["col_offset"]:2 * (o["col_offset"] + o["ncols"])].reshape(-1, 2)
            assert rel_err(h, r["H"]) < 1e-9
            w = W[2 * m * o["slot"]:2 * m * (o["slot"] + 1)].reshape(2, m).T
            assert rel_err(w, r["W"]) < 1e-9
