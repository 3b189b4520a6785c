"""Activations far below f16's range on every path that scales rows to f16 by a power of two: rows, 256-wide
pieces of rows and pixels whose largest value is 1e-30, 1e-36 or a subnormal (1e-40, and 2^-149 itself) beside
ordinary ones and zeros. The scale has to stay finite there, or zeros become NaN.

Bar: the matmul bar, 1e-3 of sum |x w|, plus what rounding the f32 result to a subnormal adds (2^-150 a piece
of 256 k or a tap, under 1e-43 here): a tiny row is held to its own size.
"""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import oracle as O
from brimkern_amd import synth
from brimkern_amd.capi import BRIK_OPT_GEMM_TILE, BRIK_OPT_PATH, BRIK_OPT_SPLITK
from helpers import Gpu, PLANES, REL_TOL
from test_gpu_conv import quantized, run as run_conv

pytestmark = pytest.mark.gpu

SUBNORMAL_SUM = 1e-43
SIZES = [1e-30, 1e-36, 1e-40, 0.0]


@pytest.fixture()
def gpu(ctx):
    g = Gpu(ctx)
    yield g
    for key in (BRIK_OPT_PATH, BRIK_OPT_SPLITK, BRIK_OPT_GEMM_TILE):
        ctx.set_option(key, 0)
    g.free()


def rows(M, K, seed):
    """Ordinary rows; in each, one 256-wide piece of a small size (zeros every third value); in row 1 all but
    the smallest subnormal are zero, and the later ones of every four rows are small as a whole."""
    x = synth.normal(seed, M * K).reshape(M, K)
    for m in range(M):
        size = np.float32(SIZES[m % 4])
        at = slice(0, K) if m >= 4 else slice((K - 1) // 256 * 256 if m % 2 else 0, K if m % 2 else 256)
        x[m, at] *= size
        x[m, at][::3] = 0
    if M > 1:
        x[1] = 0
        x[1, K - 1] = np.float32(2.0 ** -149)
    return x


def check(y, r, den):
    assert np.isfinite(y).all()
    err = np.abs(y.astype(np.float64) - r)
    assert np.all(err <= REL_TOL * den + SUBNORMAL_SUM), float((err / np.maximum(den, 1e-300)).max())


# the few-row GEMM's tiles (8, 16, 32, 64 rows; a last piece of 32 and of 160), the split-K kernel's and a
# tiled launch's rows by one wave (K <= 2048) and one block each, and rows read twice
@pytest.mark.parametrize("fmt", ["q8", "q4", "q3"])
@pytest.mark.parametrize("M,K,N,splitk,tile", [
    (6, 544, 33, 3, 0), (12, 1056, 65, 3, 0), (12, 416, 65, 3, 0), (30, 1312, 130, 3, 0), (61, 544, 70, 3, 0),
    (9, 544, 40, 2, 0), (33, 1312, 40, 2, 0),
    (9, 544, 40, 0, 8), (33, 1312, 40, 0, 8), (33, 2592, 40, 0, 8), (9, 8224, 33, 0, 8), (70, 1312, 64, 0, 13),
])
def test_matmul_rows(gpu, fmt, M, K, N, splitk, tile):
    t = synth.tensor(fmt, 70 + M, N, K)
    x = rows(M, K, 71 + M)
    r, den = getattr(O, f"matmul_t_{fmt}")(x.ravel(), *[t[k] for k in PLANES[fmt]], M, K, N, absden=True)
    gpu.ctx.set_option(BRIK_OPT_PATH, 2)
    gpu.ctx.set_option(BRIK_OPT_SPLITK, splitk)
    gpu.ctx.set_option(BRIK_OPT_GEMM_TILE, tile)
    check(gpu.matmul(fmt, x.ravel(), gpu.planes(fmt, t), M, K, N), r, den)
    assert gpu.ctx.last_kernel() == ("gemm" if tile else {2: "gemm_sk", 3: "gemm_few"}[splitk])


def test_fragment_rows(gpu):
    """The fragment GEMM's staging, 8 rows a block: a slice of the rows against the oracle."""
    M, K, N = 2045, 2560, 1024
    t = synth.tensor("q4", 80, N, K)
    x = rows(M, K, 81)
    y = gpu.matmul("q4", x.ravel(), gpu.planes("q4", t), M, K, N)
    assert gpu.ctx.last_kernel() == "gemm_frag"
    r, den = O.matmul_t_q4(np.ascontiguousarray(x[:16]).ravel(), t["nib"], t["sc"], t["mn"], 16, K, N, absden=True)
    assert np.isfinite(y).all()
    check(y[:16], r, den)


@pytest.mark.parametrize("M,K,N,splitk,tile,kernel", [
    (7, 544, 33, 3, 0, "gemm_few"), (30, 1312, 130, 3, 0, "gemm_few"), (200, 1312, 129, 0, 0, "gemm_h"),
    (100, 6176, 65, 0, 0, "gemm_h"), (40, 544, 64, 0, 5, "gemm_f16")])
def test_f16_rows(gpu, M, K, N, splitk, tile, kernel):
    rng = np.random.default_rng(M + K)
    w = (rng.standard_normal((N, K)) * 0.05).astype(np.float16).view(np.uint16)
    x = rows(M, K, 90 + M)
    r, den = O.matmul_t_f16w(x.ravel(), w.ravel(), M, K, N)
    gpu.ctx.set_option(BRIK_OPT_SPLITK, splitk)
    gpu.ctx.set_option(BRIK_OPT_GEMM_TILE, tile)
    yb = gpu.up(np.full(M * N, np.nan, np.float32))
    gpu.ctx.matmul_t_f16w(gpu.up(x), gpu.up(w), yb, M, K, N)
    assert gpu.ctx.last_kernel() == kernel
    check(gpu.ctx.download(yb, np.float32, M * N).reshape(M, N), r.reshape(M, N), den.reshape(M, N))


# tap by tap (Cin a multiple of 32), im2col 3 x 3 (a forced tile) and im2col of any kernel
@pytest.mark.parametrize("fmt", ["q8", "q4"])
@pytest.mark.parametrize("shape,tile", [((64, 12, 13, 40, 3, 3, 1, 1), 0), ((544, 11, 9, 33, 3, 3, 1, 1), 0),
                                        ((64, 12, 13, 40, 3, 3, 1, 1), 13), ((8, 12, 12, 64, 4, 4, 1, 1), 0)])
def test_conv_pixels(gpu, fmt, shape, tile):
    Cin, H, W, Cout, kh, kw, st, pd = shape
    rng = np.random.default_rng(sum(shape))
    w = rng.standard_normal(Cout * Cin * kh * kw).astype(np.float32)
    blob, deq = quantized(fmt, w)
    x = rng.standard_normal((Cin, H, W)).astype(np.float32)
    x[:, 1::4, ::3] *= np.float32(1e-36)         # single faint pixels, with zero channels, beside ordinary ones
    x[::2, 1::4, ::3] = 0
    x[:, 5:9, 4:] *= np.float32(1e-40)           # and a patch that some outputs see alone
    x[1:, 10, 2] = 0
    x[0, 10, 2] = np.float32(2.0 ** -149)
    gpu.ctx.set_option(BRIK_OPT_GEMM_TILE, tile)
    y = run_conv(gpu, fmt, x, blob, w.size, None, shape, 2)
    assert gpu.ctx.last_kernel() == ("gemm" if tile or Cin % 32 else "gemm_conv")
    wt = torch.from_numpy(np.asarray(deq, dtype=np.float64).reshape(Cout, Cin, kh, kw))
    xt = torch.from_numpy(x.astype(np.float64))[None]
    check(y, F.conv2d(xt, wt, stride=st, padding=pd)[0].numpy(),
          F.conv2d(xt.abs(), wt.abs(), stride=st, padding=pd)[0].numpy())
