"""The K-quant GEMM (csrc/kquant_gemm.hip, m > 4) against the C oracle.

Its super-block sums are exact integers, so an output differs from the oracle's
double sums by f32 rounding only: about nsb + 4 roundings of 2^-24 of the summed
magnitude, itself about sqrt(nsb) of the largest output for these inputs: 5e-6
at nsb = 16 (f32 y). bf16 y adds half a step of its 8-bit significand: at
most 2^-8 of the value.
"""
import numpy as np
import pytest
from test_gpu_kquant import ctx, dev, encode, make_weight, note, oracle_y, torch  # noqa: F401

pytestmark = pytest.mark.gpu

TOL = {"f32": 5e-6, "bf16": 5e-6 + 2.0 ** -8}

# m, out, in: the tiles the planner takes at 256 CUs, their row and column
# remainders, super-block counts that do not fill a step, the smallest shapes
SHAPES = [(5, 16, 256), (5, 4099, 1280), (16, 37, 512), (17, 3001, 1024), (33, 130, 768), (44, 4663, 512),
          (64, 11008, 512), (65, 1031, 2304), (100, 3000, 1024), (129, 5000, 512), (200, 2050, 256), (257, 11008, 512), (511, 6001, 256)]


def run(torch, ctx, orc, fmt, arrs, m, out, in_, x, ydt="f32"):  # noqa: F811
    """(rq_qmatmul, rq_qmatmul_q8k, oracle rows' reference, rows)"""
    import raster_amd

    sub = 32 if fmt == "q4k" else 16
    w = make_weight(raster_amd, ctx, fmt, arrs, out, in_)
    xt = dev(torch, x)
    dt = torch.bfloat16 if ydt == "bf16" else torch.float32
    xq, xs, bs = raster_amd.quantize_act_q8k(ctx, xt, in_, sub)
    y2 = w.matmul_q8k(xq, xs, bs, out_dtype=dt)
    y1 = w.matmul(xt, out_dtype=dt)
    torch.cuda.synchronize()
    w.destroy()
    rows = np.unique(np.concatenate([np.arange(min(out, 40)), np.arange(max(0, out - 40), out),
                                     np.random.default_rng(out).integers(0, out, 40)]))
    rq, rs, rb = orc.quantize_act_q8k(x, m, in_, sub)
    return y1.float().cpu().numpy(), y2.float().cpu().numpy(), oracle_y(orc, fmt, arrs, rq, rs, rb, m, in_, out,
                                                                        rows), rows


@pytest.mark.parametrize("ydt", ["f32", "bf16"])
@pytest.mark.parametrize("fmt", ["q4k", "q6k"])
@pytest.mark.parametrize("m,out,in_", SHAPES)
def test_kquant_gemm(torch, ctx, orc, fmt, m, out, in_, ydt):  # noqa: F811
    note(f"K-quant GEMM {fmt} m={m} {out}x{in_} y={ydt}")
    x = np.random.default_rng(m + in_).standard_normal(m * in_).astype(np.float32)
    y1, y2, ref, rows = run(torch, ctx, orc, fmt, encode(orc, fmt, out, in_, seed=m), m, out, in_, x, ydt)
    assert np.array_equal(y1, y2)  # packed and row-major activations: the same sums
    assert np.abs(y1[:, rows] - ref).max() <= TOL[ydt] * np.abs(ref).max()


@pytest.mark.parametrize("fmt", ["q4k", "q6k"])
def test_kquant_gemm_extreme_codes(torch, ctx, orc, fmt):  # noqa: F811
    """The largest digits: every code, sub-block scale and activation at its bound."""
    m, out, in_ = 20, 48, 512
    note(f"K-quant GEMM extremes {fmt}")
    n = out * in_
    rng = np.random.default_rng(3)
    sign = rng.choice([-1.0, 1.0], size=(out, in_ // 256)).astype(np.float32).ravel()
    if fmt == "q4k":
        arrs = (np.full(n // 2, 0xFF, np.uint8), sign * 1e-3, sign * 2e-3, np.full(n // 32, 63, np.uint8),
                rng.choice([-128, 127], size=n // 32).astype(np.int8))
    else:
        arrs = (rng.choice([0, 63], size=n).astype(np.uint8), rng.choice([-128, 127], size=n // 16).astype(np.int8),
                sign * 1e-4)
    x = np.where(rng.random((m, 1)) < 0.5, 1.0, -1.0).astype(np.float32).repeat(in_, 1).ravel()
    y1, y2, ref, rows = run(torch, ctx, orc, fmt, arrs, m, out, in_, x)
    assert np.array_equal(y1, y2)
    assert np.abs(y1[:, rows] - ref).max() <= TOL["f32"] * np.abs(ref).max()


@pytest.mark.parametrize("case", ["aq", "inf"])
def test_kquant_gemm_refused_scales(torch, ctx, orc, case):  # noqa: F811
    """aq above 6 bits or a scale that is not finite keeps the GEMV: the rows of
    a 20-row call equal the same rows in calls of four, bit for bit."""
    import raster_amd

    m, out, in_ = 20, 64, 512
    note(f"K-quant GEMM refused scales {case}")
    wq, da, db, aq, bq = (a.copy() for a in encode(orc, "q4k", out, in_, seed=9))
    if case == "aq":
        aq[5] = 200
    else:
        da[7] = np.inf
    w = make_weight(raster_amd, ctx, "q4k", (wq, da, db, aq, bq), out, in_)
    x = dev(torch, np.random.default_rng(1).standard_normal((m, in_)).astype(np.float32))
    y = w.matmul(x).cpu().numpy()
    parts = np.concatenate([w.matmul(x[i:i + 4].contiguous()).cpu().numpy() for i in range(0, m, 4)])
    w.destroy()
    assert np.array_equal(y.view(np.uint32), parts.view(np.uint32))


@pytest.mark.parametrize("fmt", ["q4k", "q6k"])
def test_kquant_gemm_special_activations(torch, ctx, orc, fmt):  # noqa: F811
    """A row with an infinite activation is NaN, a zero row zero; the other rows do not change."""
    import raster_amd

    m, out, in_ = 40, 300, 512
    note(f"K-quant GEMM special activations {fmt}")
    w = make_weight(raster_amd, ctx, fmt, encode(orc, fmt, out, in_, seed=4), out, in_)
    x = np.random.default_rng(2).standard_normal((m, in_)).astype(np.float32)
    y0 = w.matmul(dev(torch, x)).cpu().numpy()
    x[3, 7] = np.inf
    x[39, 300] = -np.inf
    x[17] = 0.0
    y = w.matmul(dev(torch, x)).cpu().numpy()
    w.destroy()
    assert np.isnan(y[[3, 39]]).all() and (y[17] == 0).all()
    keep = np.setdiff1d(np.arange(m), [3, 17, 39])
    assert np.array_equal(y[keep], y0[keep])
