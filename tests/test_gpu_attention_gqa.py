"""rq_decode_attention on long caches (the grouped-query kernel and the wide
merge, csrc/attention.hip) against the same step in 64 bits.

Scores and values are f32: a score's head_dim products and their sum err by at
most (head_dim + 8) 2^-24 |q| |k| scale, about 2e-6 for N(0, 1) rows, which the
exponential passes on, and the weighted sum adds (rows' tree, <= 64 terms in a
row) 2^-24 each: 1e-5 of the largest output bounds both.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t

    if not t.cuda.is_available():
        pytest.skip("no GPU")
    return t


@pytest.fixture(scope="module")
def ctx(torch):
    import raster_amd

    c = raster_amd.Context(0)
    yield c
    c.close()


def rope(torch, t, hd, pos):
    ang = pos * torch.exp(torch.arange(hd // 2, dtype=torch.float64, device="cuda") * (-2.0 / hd) * np.log(1e4))
    a, b = t[:, :hd // 2], t[:, hd // 2:]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], 1)


# heads, KV heads, head_dim, cached rows: 1, 2, 4 and 8 heads per KV head at each
# lanes-per-row width, partial vectors, ranges and chunks that do not divide,
# either side of the planner's line, 16 to 64 ranges; then many heads: one range
# (two cases), 2, 2, 4, 8 and 10 of them, and two cases below their line
CASES = [(32, 8, 128, 4096), (32, 8, 128, 1021), (64, 8, 128, 1999), (16, 2, 64, 9001), (16, 16, 128, 2050),
         (24, 12, 128, 1500), (32, 8, 64, 2049), (12, 12, 64, 5463), (8, 4, 256, 2100), (16, 4, 256, 1100),
         (8, 8, 512, 1100), (16, 2, 100, 5300), (16, 4, 36, 8000), (64, 8, 128, 767), (32, 8, 128, 300),
         (256, 256, 128, 130), (256, 256, 128, 200), (512, 128, 64, 140), (128, 128, 128, 800), (256, 32, 128, 200),
         (64, 32, 128, 777), (96, 24, 128, 600), (96, 96, 128, 600), (144, 72, 128, 230)]


@pytest.mark.parametrize("nq,nkv,hd,pos", CASES)
def test_long_cache(torch, ctx, nq, nkv, hd, pos):
    import raster_amd

    print(f"[gpu] attention {nq}/{nkv}x{hd} pos={pos}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(pos)
    q, k, v = (torch.randn(n * hd, generator=g, device="cuda") for n in (nq, nkv, nkv))
    kc, vc = (torch.randn((pos + 1, nkv * hd), generator=g, device="cuda") for _ in range(2))
    kc[pos // 3] *= 4.0  # a peaked row
    scale = hd ** -0.5
    kr, vr = kc.double(), vc.double()
    kr[pos], vr[pos] = rope(torch, k.double().view(nkv, hd), hd, pos).view(-1), v.double()
    qr = rope(torch, q.double().view(nq, hd), hd, pos)
    out = raster_amd.decode_attention(ctx, q, k, v, kc, vc, pos, nq, nkv, hd, 1e4, scale).view(nq, hd)
    for h in range(nq):
        j = h // (nq // nkv)
        p = torch.softmax(kr[:, j * hd:(j + 1) * hd] @ qr[h] * scale, 0)
        ref = p @ vr[:, j * hd:(j + 1) * hd]
        assert float((out[h].double() - ref).abs().max()) <= 1e-5 * float(ref.abs().max())
    assert torch.equal(vc[pos], v) and float((kc[pos].double() - kr[pos]).abs().max()) < 1e-6


@pytest.mark.parametrize("nq,nkv,pos", [(32, 8, 2000), (256, 256, 200)])
def test_infinite_scores(torch, ctx, nq, nkv, pos):
    """A key of +inf: a head whose score is +inf is NaN (inf - inf, as in the
    reference's softmax), one whose score is -inf leaves the row out."""
    import raster_amd

    hd, row = 128, pos // 2
    print(f"[gpu] attention infinite key {nq}/{nkv} pos={pos}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(2)
    q, k, v = (torch.randn(n * hd, generator=g, device="cuda") for n in (nq, nkv, nkv))
    kc, vc = (torch.randn((pos + 1, nkv * hd), generator=g, device="cuda") for _ in range(2))
    kc[row, 5::hd] = float("inf")
    out = raster_amd.decode_attention(ctx, q, k, v, kc, vc, pos, nq, nkv, hd, 1e4, hd ** -0.5).view(nq, hd)
    qr, keep = rope(torch, q.double().view(nq, hd), hd, pos), torch.arange(pos + 1, device="cuda") != row
    neg = 0
    for h in range(nq):
        if float(qr[h, 5]) > 0:
            assert bool(torch.isnan(out[h]).all())
            continue
        j = h // (nq // nkv)
        p = torch.softmax(kc[keep, j * hd:(j + 1) * hd].double() @ qr[h] * hd ** -0.5, 0)
        ref = p @ vc[keep, j * hd:(j + 1) * hd].double()
        assert float((out[h].double() - ref).abs().max()) <= 1e-5 * float(ref.abs().max())
        neg += 1
    assert 0 < neg < nq


def test_nan_scores(torch, ctx):
    """A NaN key makes its head's outputs NaN; the other heads are as before."""
    import raster_amd

    nq, nkv, hd, pos = 32, 8, 128, 2000
    print("[gpu] attention NaN row", flush=True)
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.randn(n * hd, generator=g, device="cuda") for n in (nq, nkv, nkv))
    kc, vc = (torch.randn((pos + 1, nkv * hd), generator=g, device="cuda") for _ in range(2))
    args = (pos, nq, nkv, hd, 1e4, hd ** -0.5)
    a = raster_amd.decode_attention(ctx, q, k, v, kc, vc, *args).view(nkv, -1).clone()
    kc[777, 3 * hd + 5] = float("nan")
    b = raster_amd.decode_attention(ctx, q, k, v, kc, vc, *args).view(nkv, -1)
    keep = [i for i in range(nkv) if i != 3]
    assert bool(torch.isnan(b[3]).all()) and torch.equal(a[keep], b[keep])
