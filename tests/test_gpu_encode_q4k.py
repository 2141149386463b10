"""rq_q4k_of bit for bit against the oracle where the wave's shared reads have
edges: rows shorter than a super-block, padded tails of every kind, a number of
super-blocks that does not fill a wave's eight or a workgroup's 32, element-wise
reads (in % 4 != 0, W off 16-byte alignment)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("out,in_", [(1, 1), (1, 4), (3, 31), (9, 32), (5, 252), (33, 256), (7, 260), (3, 1001),
                                     (11, 2044), (4, 4000), (65, 513)])
def test_q4k_of_edges(orc, out, in_, offset):
    import torch

    import raster_amd

    print(f"[gpu] q4k_of {out}x{in_} offset {offset}", flush=True)
    rng = np.random.default_rng(out * in_)
    W = (rng.standard_normal(out * in_) * 0.05).astype(np.float32)
    W[: min(W.size, 40)] = 0.0
    buf = torch.zeros(W.size + 8, device="cuda")
    t = buf[offset:offset + W.size]
    t.copy_(torch.from_numpy(W))
    with raster_amd.Context(0) as ctx:
        got = raster_amd.q4k_of(ctx, t, out, in_)
        torch.cuda.synchronize()
    ref = orc.q4k_of(W, out, in_)
    for name, r in zip(("wq", "da", "db", "aq", "bq"), ref):
        g = got[name].cpu().numpy()
        assert np.array_equal(g.view(np.uint8), np.asarray(r).ravel().view(np.uint8)), name
    assert got["in"] == ref[5]
