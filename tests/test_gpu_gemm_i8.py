"""The int8-activation GEMM (csrc/gemm.hip, m > 16) against 64-bit products of
the quantized activations and the dequantized weight: the block dots are exact,
each block adds its product of scales (one rounding), its product with the dot
and the sum's rounding: |y - ref| <= (in / 32 + 8) 2^-23 sum_b |ws xs dot_b|, and
2^-8 |y| more for bf16 y.
"""
import numpy as np
import pytest
from test_gpu_gemm_f32 import ctx, rows, torch, weight  # noqa: F401

pytestmark = pytest.mark.gpu

# the tiles (32 x 32, 128 x 64, 128 x 128) with row, column and K-step remainders
SHAPES = [(17, 3, 32), (18, 4100, 96), (40, 300, 1056), (129, 4099, 416), (300, 2050, 224), (256, 11008, 160),
          (200, 30001, 288)]


@pytest.mark.parametrize("fmt,ydt", [("q8", "f32"), ("q4h", "f32"), ("q4f", "bf16")])
@pytest.mark.parametrize("m,out,in_", SHAPES)
def test_gemm_i8(torch, ctx, m, out, in_, fmt, ydt):  # noqa: F811
    import raster_amd

    print(f"[gpu] int8 GEMM {fmt} m={m} {out}x{in_} y={ydt}", flush=True)
    w = weight(ctx, fmt, out, in_, m)
    x = rows(torch, m, in_, out)
    x[2] = 0.0
    xq, xs, xsum = raster_amd.quantize_act_i8(ctx, x, in_)
    y = w.matmul_i8(xq, xs, xsum, out_dtype=torch.bfloat16 if ydt == "bf16" else torch.float32).double()
    W = w.dequant().double()
    w.destroy()
    ref, mag = torch.zeros_like(y), torch.zeros_like(y)
    for b in range(in_ // 32):
        k = slice(32 * b, 32 * b + 32)
        d = (xq[:, k].double() * xs[:, b:b + 1].double()) @ W[:, k].T
        ref += d
        mag += d.abs()
    bound = (in_ / 32 + 8) * 2.0 ** -23 * mag + (2.0 ** -8 * ref.abs() if ydt == "bf16" else 0.0)
    # the dequantized weight is scale * code rounded to f32: one more rounding of the operands
    assert bool(((y - ref).abs() <= bound + 2.0 ** -23 * (x.abs().double() @ W.abs().T)).all())


@pytest.mark.parametrize("m,out,in_", [(18, 40, 96), (129, 4099, 160), (200, 30001, 288)])
def test_gemm_i8_infinite_tail_scale(torch, ctx, m, out, in_):  # noqa: F811
    """An infinite activation scale of the last block makes its row's outputs
    infinite, also where the blocks do not fill the kernel's steps."""
    import raster_amd

    print(f"[gpu] int8 GEMM infinite tail m={m} {out}x{in_}", flush=True)
    w = raster_amd.QWeight.q8(np.full(out * in_, 127, np.int8), np.full(out * in_ // 32, 0.01, np.float32), out, in_,
                              ctx)
    xq, xs, xsum = raster_amd.quantize_act_i8(ctx, torch.ones((m, in_), device="cuda"), in_)
    xs[3:, -1] = float("inf")
    y = w.matmul_i8(xq, xs, xsum)
    w.destroy()
    assert bool(torch.isfinite(y[:3]).all()) and bool((y[3:] == float("inf")).all())


@pytest.mark.parametrize("fmt,out,in_", [("q4f", 35, 2 ** 24 + 96), ("q8", 1, 2 ** 26)])
def test_gemm_i8_long_rows(torch, ctx, fmt, out, in_):  # noqa: F811
    """Rows whose packed activations pass 32-bit offsets (2^26: 4 GiB of codes, then
    their scales): codes of -1, 0 and 1 and scales of 1 and 2, y an exact integer."""
    import raster_amd

    m = 17
    print(f"[gpu] int8 GEMM long rows {fmt} {out}x{in_}", flush=True)
    rng = np.random.default_rng(in_)
    scales = np.ones(out * in_ // 32, np.float32)
    if fmt == "q8":
        w = raster_amd.QWeight.q8(rng.integers(-1, 2, out * in_, dtype=np.int8), scales, out, in_, ctx)
    else:
        nib = rng.integers(7, 10, out * in_ // 2, dtype=np.uint8)
        w = raster_amd.QWeight.q4(nib | (rng.integers(7, 10, out * in_ // 2, dtype=np.uint8) << 4), scales, out, in_,
                                  ctx)
    g = torch.Generator(device="cuda").manual_seed(2)
    xq = torch.randint(-1, 2, (m, in_), generator=g, device="cuda", dtype=torch.int8)
    xs = torch.randint(1, 3, (m, in_ // 32), generator=g, device="cuda").float()
    xsum = xq.view(m, -1, 32).sum(2, dtype=torch.int32)
    y = w.matmul_i8(xq, xs, xsum)
    W = w.dequant()
    w.destroy()
    for t in (0, 7, 16):
        x = (xq[t].view(-1, 32).float() * xs[t].view(-1, 1)).view(-1)
        for o in range(out):
            assert float(y[t, o]) == float((x * W[o]).sum(dtype=torch.float64)), (t, o)
