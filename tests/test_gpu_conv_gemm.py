"""The tap-by-tap convolution GEMM (channel counts that are multiples of 32, up to 25 taps) against the f64
convolution of the dequantized weights: one and several 32-channel steps per tap, more than one staging round
(Cin > 512), ragged channel and pixel tiles, slices of the sum, taps outside the image on every side, strides.

Tolerance: f16 operands (2^-11 each, relative to the operand: every pixel row has its own scale) and f32 sums,
so 2^-10 + K 2^-24 of sum |x w|.
"""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from brimkern_amd import layout
from brimkern_amd.capi import BRIK_OPT_PATH, Context
from helpers import Gpu, PLANES
from test_gpu_conv import quantized, run

pytestmark = pytest.mark.gpu


@pytest.fixture()
def gpu(ctx):
    g = Gpu(ctx)
    yield g
    g.free()
    ctx.set_option(BRIK_OPT_PATH, 0)


SHAPES = [
    (32, 8, 8, 16, 1, 1, 1, 0),        # one step in all
    (512, 8, 8, 1, 1, 1, 1, 0),        # one output channel
    (512, 9, 9, 40, 1, 1, 1, 0),       # pixel rows that just fit the im2col rows' room
    (32, 9, 11, 33, 3, 3, 1, 1),       # one step per tap
    (64, 17, 15, 65, 3, 3, 2, 1),      # stride 2, every tile ragged
    (96, 12, 13, 16, 5, 5, 1, 2),      # 25 taps, sliced sum
    (544, 9, 9, 40, 3, 3, 1, 1),       # two staging rounds of channels
    (32, 6, 40, 130, 1, 25, 1, 12),    # a 1 x 25 kernel, pad also above and below
    (64, 16, 16, 130, 3, 3, 1, 3),     # pad wider than the kernel's reach
    (160, 40, 40, 300, 3, 3, 1, 1),    # many tiles
]


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("fmt", ["q8", "q4"])
@pytest.mark.parametrize("shape", SHAPES, ids=[f"{s[0]}x{s[1]}x{s[2]}-{s[3]}-k{s[4]}x{s[5]}s{s[6]}p{s[7]}" for s in SHAPES])
def test_conv_gemm(gpu, fmt, bias, shape):
    Cin, H, W, Cout, kh, kw, st, pd = shape
    rng = np.random.default_rng(sum(shape))
    w = rng.standard_normal(Cout * Cin * kh * kw).astype(np.float32)
    blob, deq = quantized(fmt, w)
    # pixels of very different magnitudes: every tap is scaled by its own pixel
    x = (rng.standard_normal((Cin, H, W)) * 2.0 ** rng.integers(-20, 20, (1, H, W))).astype(np.float32)
    b = rng.standard_normal(Cout).astype(np.float32) if bias else None
    y = run(gpu, fmt, x, blob, w.size, b, shape, 2).astype(np.float64)
    assert gpu.ctx.last_kernel() == "gemm_conv"
    wt = torch.from_numpy(np.asarray(deq, dtype=np.float64).reshape(Cout, Cin, kh, kw))
    xt = torch.from_numpy(x.astype(np.float64))[None]
    ref = F.conv2d(xt, wt, stride=st, padding=pd)[0].numpy()
    den = F.conv2d(xt.abs(), wt.abs(), stride=st, padding=pd)[0].numpy()
    if bias:
        ref = ref + b[:, None, None]
        den = den + np.abs(b)[:, None, None]
    tol = 2.0 ** -10 + Cin * kh * kw * 2.0 ** -24
    assert np.all(np.abs(y - ref) <= tol * den)


# weight fragments behind the pixel rows, and past the im2col rows' size (a buffer of their own)
@pytest.mark.parametrize("shape", [(32, 40, 40, 40, 3, 3, 1, 1), (256, 8, 8, 200, 3, 3, 1, 1), (512, 8, 8, 64, 1, 1, 1, 0)],
                         ids=["behind", "apart", "apart1x1"])
def test_recorded_conv_runs_the_eager_kernel(shape):
    """A convolution recorded before it ever ran eagerly, on workspaces that another one left, gives the bits of
    the eager call, also replayed after larger eager calls."""
    Cin, H, W, Cout, kh, kw, st, pd = shape
    rng = np.random.default_rng(sum(shape))
    blob, _ = quantized("q4", rng.standard_normal(Cout * Cin * kh * kw).astype(np.float32))
    n, pixels = Cout * Cin * kh * kw, H * W
    with Context(0) as c:
        gpu = Gpu(c)
        buf, xb = gpu.up(blob), gpu.up(rng.standard_normal(Cin * H * W).astype(np.float32))
        planes = [buf.offset(layout.plane_offsets("q4", n)[p][0]) for p in PLANES["q4"]]
        y = gpu.up(np.zeros(Cout * pixels, np.float32))

        def other(side):
            b, _ = quantized("q4", rng.standard_normal(32 * 32 * 9).astype(np.float32))
            run(gpu, "q4", rng.standard_normal((32, side, side)).astype(np.float32), b, 32 * 32 * 9, None,
                (32, side, side, 32, 3, 3, 1, 1), 0)

        def bits():
            r = c.download(y, np.uint32, Cout * pixels)
            c.h2d(y, np.zeros(Cout * pixels, np.float32))
            return r

        other(64)                               # 2.1 MB of im2col rows
        c.graph_begin()
        c.conv2d("q4", xb, planes, None, y, *shape)
        assert c.last_kernel() == "gemm_conv"
        g = c.graph_end()
        g.launch()
        recorded = bits()
        c.conv2d("q4", xb, planes, None, y, *shape)
        assert c.last_kernel() == "gemm_conv"
        assert np.array_equal(bits(), recorded) and recorded.any()
        for _ in range(3):
            other(40)
            g.launch()
            assert np.array_equal(bits(), recorded)
        g.destroy()
        gpu.free()
