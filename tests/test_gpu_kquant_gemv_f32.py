"""K-quant GEMV that quantizes a short f32 x itself: bit for bit the q8_K
quantizer followed by the GEMV on its output, around the line of m * in = 12288,
for workgroups of every wave count, partial row groups and padded activation
rows, non-finite and zero super-blocks, and for a y that overlaps x."""
import ctypes as C

import numpy as np
import pytest
from test_gpu_kquant import ctx, dev, encode, make_weight, note, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def both(torch, ctx, w, fmt, x, ydt):
    import raster_amd

    y1 = w.matmul(x, out_dtype=ydt)
    xq, xs, bs = raster_amd.quantize_act_q8k(ctx, x, x.shape[1], 32 if fmt == "q4k" else 16)
    y2 = w.matmul_q8k(xq, xs, bs, out_dtype=ydt)
    torch.cuda.synchronize()
    return y1.float().cpu().numpy(), y2.float().cpu().numpy()


@pytest.mark.parametrize("fmt", ["q4k", "q6k"])
@pytest.mark.parametrize("m,out,in_", [(1, 1, 256), (1, 37, 1024), (1, 1501, 4096), (1, 14336, 4096), (1, 33, 12288),
                                       (1, 33, 12544), (2, 1030, 5888), (2, 9000, 6144), (2, 65, 6400), (3, 517, 4096),
                                       (4, 700, 3072), (4, 515, 3328), (4, 2049, 256)])
def test_fused_quantizer_bits(torch, ctx, orc, fmt, m, out, in_):
    import raster_amd

    note(f"K-quant fused GEMV {fmt} m={m} {out}x{in_}")
    # the bits do not depend on what the codes are: few encoded rows, tiled
    rows = min(out, 64)
    few = encode(orc, fmt, rows, in_, seed=out + m)
    arrs = tuple(np.resize(a.reshape(rows, -1), (out, a.size // rows)).ravel() for a in few)
    w = make_weight(raster_amd, ctx, fmt, arrs, out, in_)
    try:
        x = np.random.default_rng(in_ + m).standard_normal((m, in_)).astype(np.float32)
        x[:, :256] *= np.float32(1e-30)
        if in_ > 256:
            x[m - 1, 256:512] = 0.0
        for ydt in (torch.float32, torch.bfloat16):
            a, b = both(torch, ctx, w, fmt, dev(torch, x), ydt)
            assert np.all(np.isfinite(a)) and np.array_equal(a.view(np.uint32), b.view(np.uint32))
        x[0, 3], x[m - 1, in_ - 1] = np.inf, np.nan
        a, b = both(torch, ctx, w, fmt, dev(torch, x), torch.float32)
        assert np.array_equal(a, b, equal_nan=True)
    finally:
        w.destroy()


@pytest.mark.parametrize("fmt", ["q4k", "q6k"])
def test_y_over_x(torch, ctx, orc, fmt):
    # y in the buffer of x: x has to be read whole before any y is stored
    import raster_amd
    from raster_amd import _lib

    n = 4096
    few = encode(orc, fmt, 64, n, seed=3)
    arrs = tuple(np.resize(a.reshape(64, -1), (n, a.size // 64)).ravel() for a in few)
    w = make_weight(raster_amd, ctx, fmt, arrs, n, n)
    try:
        buf = dev(torch, np.random.default_rng(4).standard_normal((2, n)).astype(np.float32))
        ref = w.matmul(buf[:1].clone())
        for off in (0, n // 2):  # the same rows, and the upper half of x with what follows it
            b = buf.clone().view(-1)
            _lib.call("rq_qmatmul", ctx.handle, w.handle, C.c_void_p(b.data_ptr()), _lib.RQ_F32,
                      C.c_void_p(b.data_ptr() + 4 * off), _lib.RQ_F32, 1,
                      C.c_void_p(torch.cuda.current_stream().cuda_stream))
            torch.cuda.synchronize()
            assert torch.equal(b[off:off + n], ref.view(-1))
    finally:
        w.destroy()
