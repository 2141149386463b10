"""The f32-activation GEMM (csrc/gemm.hip, m > 16) against 64-bit products of
the dequantized weight.

x enters as two bf16 terms (|x - hi - lo| <= 2^-17 |x|), products and codes are
exact, the sums f32: |y - ref| <= (2^-17 + (in / 32 + 64) 2^-24) sum |x w| (a
block's 64 terms, then one FMA per block and the K-slices' sums), and 2^-8 |y|
more for bf16 y.
"""
import numpy as np
import pytest

from raster_amd import workloads as wl

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


def weight(ctx, fmt, out, in_, seed):
    import raster_amd

    if fmt == "q8":
        return raster_amd.QWeight.q8(*wl.q8_weights(out, in_, seed), out, in_, ctx)
    p, s = wl.q4_weights(out, in_, seed)
    return raster_amd.QWeight.q4(p, s if fmt == "q4h" else s.view(np.float16).astype(np.float32), out, in_, ctx)


def rows(torch, m, in_, seed):
    return torch.from_numpy(wl.activations(m, in_, seed)).cuda().view(m, in_)


# m, out, in: each tile of the planner at 256 CUs (32 x 32, 64 x 32, 128 x 64,
# 128 x 96, 128 x 192) with row, column and K-step remainders, the smallest calls
SHAPES = [(17, 1, 32), (17, 40, 96), (33, 1000, 1056), (64, 4099, 416), (70, 8000, 1024), (200, 3000, 2080),
          (129, 11008, 160), (300, 5000, 672), (130, 20003, 288), (333, 11008, 1024), (257, 24000, 352)]


@pytest.mark.parametrize("fmt,ydt", [("q8", "f32"), ("q4h", "bf16"), ("q4f", "f32"), ("q8", "bf16")])
@pytest.mark.parametrize("m,out,in_", SHAPES)
def test_gemm_f32(torch, ctx, m, out, in_, fmt, ydt):
    print(f"[gpu] f32 GEMM {fmt} m={m} {out}x{in_} y={ydt}", flush=True)
    w = weight(ctx, fmt, out, in_, m)
    x = rows(torch, m, in_, out)
    y = w.matmul(x, out_dtype=torch.bfloat16 if ydt == "bf16" else torch.float32).double()
    W = w.dequant().double()
    w.destroy()
    ref, mag = x.double() @ W.T, x.double().abs() @ W.abs().T
    bound = (2.0 ** -17 + (in_ / 32 + 64) * 2.0 ** -24) * mag + (2.0 ** -8 * ref.abs() if ydt == "bf16" else 0.0)
    assert bool(((y - ref).abs() <= bound).all())


@pytest.mark.parametrize("m,out,in_", [(40, 300, 1056), (130, 20003, 288), (333, 11008, 512), (64, 4099, 416)])
def test_gemm_f32_without_scratch(torch, m, out, in_):
    """A first call under graph capture has no scratch and reads x itself: the
    same bits as the eager call, on every replay."""
    import raster_amd

    print(f"[gpu] f32 GEMM captured first m={m} {out}x{in_}", flush=True)
    with raster_amd.Context(0) as c:
        w = weight(c, "q8", out, in_, 3)
        x = rows(torch, m, in_, 5)
        y = torch.empty((m, out), device="cuda")
        s = torch.cuda.Stream()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            w.matmul(x, y=y)
        ref = w.matmul(x)
        for i in range(3):
            y.fill_(float("nan"))
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, ref)
            w.matmul(x * (i + 2))
        w.destroy()


def test_gemm_f32_row_chunks(torch, ctx):
    """A call past one packed copy's rows runs in chunks: the rows' results do not change."""
    m, out, in_ = 600, 70, 32768
    print("[gpu] f32 GEMM row chunks", flush=True)
    w = weight(ctx, "q8", out, in_, 1)
    x = rows(torch, m, in_, 2)
    y = w.matmul(x)
    W = w.dequant().double()
    ref, mag = x.double() @ W.T, x.double().abs() @ W.abs().T
    w.destroy()
    assert bool(((y.double() - ref).abs() <= (2.0 ** -17 + (in_ / 32 + 64) * 2.0 ** -24) * mag).all())


@pytest.mark.parametrize("m,out,in_", [(20, 64, 96), (150, 11008, 160)])
def test_gemm_f32_special_rows(torch, ctx, m, out, in_):
    """inf and NaN make their row not finite, a zero row zero; the other rows do not change."""
    print(f"[gpu] f32 GEMM special rows m={m}", flush=True)
    w = weight(ctx, "q4f", out, in_, 4)
    x = rows(torch, m, in_, 6)
    y0 = w.matmul(x)
    x[1, 5], x[m - 1, in_ - 1], x[7] = float("inf"), float("nan"), 0.0
    y = w.matmul(x)
    w.destroy()
    keep = [i for i in range(m) if i not in (1, 7, m - 1)]
    assert not bool(torch.isfinite(y[[1, m - 1]]).any()) and bool((y[7] == 0).all()) and torch.equal(y[keep], y0[keep])


@pytest.mark.parametrize("m,out,in_", [(20, 64, 96), (64, 4099, 160), (200, 3000, 288), (129, 11008, 160),
                                       (130, 20003, 224)])
def test_gemm_f32_overflowing_tail(torch, m, out, in_):
    """A last block whose sum passes the largest float gives inf for finite x, also
    where the blocks do not fill the kernels' steps; with and without scratch."""
    import raster_amd

    print(f"[gpu] f32 GEMM overflowing tail m={m} {out}x{in_}", flush=True)
    with raster_amd.Context(0) as c:
        w = raster_amd.QWeight.q8(np.full(out * in_, 127, np.int8), np.full(out * in_ // 32, 0.01, np.float32), out, in_,
                                  c)
        x = torch.ones((m, in_), device="cuda")
        x[3:, in_ - 32:] = 2.0 ** 126
        y = torch.empty((m, out), device="cuda")
        s = torch.cuda.Stream()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            w.matmul(x, y=y)
        g.replay()
        for got in (y, w.matmul(x)):
            torch.cuda.synchronize()
            assert bool(torch.isfinite(got[:3]).all()) and bool((got[3:] == float("inf")).all())
        w.destroy()


@pytest.mark.parametrize("fmt,out,in_", [("q4h", 40, 2 ** 24 + 96), ("q4f", 3, 2 ** 24 + 32), ("q8", 1, 2 ** 28)])
def test_gemm_f32_long_rows(torch, ctx, fmt, out, in_):
    """Rows whose weights or activations pass 32-bit offsets (16 padded rows of 2^28
    codes are 4 GiB): x and codes of -1, 0 and 1, so that y is an exact integer."""
    import raster_amd

    m = 17
    print(f"[gpu] f32 GEMM long rows {fmt} {out}x{in_}", flush=True)
    rng = np.random.default_rng(in_)
    scales = np.ones(out * in_ // 32, np.float16 if fmt == "q4h" else np.float32)
    if fmt == "q8":
        w = raster_amd.QWeight.q8(rng.integers(-1, 2, out * in_, dtype=np.int8), scales, out, in_, ctx)
    else:
        nib = rng.integers(7, 10, out * in_ // 2, dtype=np.uint8)
        w = raster_amd.QWeight.q4(nib | (rng.integers(7, 10, out * in_ // 2, dtype=np.uint8) << 4), scales, out, in_,
                                  ctx)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randint(-1, 2, (m, in_), generator=g, device="cuda", dtype=torch.int8).float()
    y = w.matmul(x)
    W = w.dequant()
    w.destroy()
    for o in range(out):
        for t in (0, 7, 16):
            assert float(y[t, o]) == float((x[t] * W[o]).sum(dtype=torch.float64)), (t, o)
