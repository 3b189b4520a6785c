"""The fragment GEMM (gemm_frag.hip): W dequantized once into MFMA fragment order, for calls of many rows.

Its sums run in the order of the tiled GEMM, so a call that takes it must give the same bits as the same
call with a tile forced (which keeps it off that route); a few rows, the first and last among them, are
also checked against the oracle within the matmul bar, 1e-3 of sum |x w|. The shapes are ones the
runtime's cost model sends there: each of the four tiles, ragged rows and columns, K of odd group counts,
rows staged 8 and 4 at a time and read twice, and a matrix wider than one column slab.
"""
import numpy as np
import pytest

import oracle as O
from brimkern_amd import synth
from brimkern_amd.capi import BRIK_OPT_GEMM_TILE, Context
from helpers import Gpu

pytestmark = pytest.mark.gpu

SHAPES = [
    (4096, 2560, 2560, "q4"),     # 192 x 256 tiles
    (4095, 2592, 2559, "q8"),     # 192 x 256, ragged in every dimension (K of 81 groups)
    (1500, 4128, 4100, "q3"),     # 128 x 256
    (900, 4160, 4001, "q3"),      # 128 x 128
    (3713, 2432, 544, "q4"),      # few columns
    (4001, 288, 2047, "q8"),      # three steps of 128 k, the last of one group
    (829, 8608, 1688, "q3"),      # 64 x 128; rows of more than 5120 are staged 4 at a time
    (1030, 10272, 1000, "q3"),    # rows past 10240: the tail of the row is read twice
    (1100, 2560, 26500, "q3"),    # 136 MB of f16 panels: two column slabs
]


def _call(gpu, fmt, xb, planes, yb, M, K, N, tile):
    gpu.ctx.set_option(BRIK_OPT_GEMM_TILE, tile)
    try:
        getattr(gpu.ctx, "matmul_t_" + fmt)(xb, *planes, yb, M, K, N)
        assert gpu.ctx.last_kernel() == ("gemm" if tile else "gemm_frag")
    finally:
        gpu.ctx.set_option(BRIK_OPT_GEMM_TILE, 0)
    return gpu.ctx.download(yb, np.float32, M * N).reshape(M, N)


@pytest.mark.parametrize("M,K,N,fmt", SHAPES)
def test_frag_equals_tiled(ctx, M, K, N, fmt):
    gpu = Gpu(ctx)
    try:
        t = synth.tensor(fmt, 11 + M, N, K)
        x = synth.normal(5 + M, M * K).reshape(M, K)
        x *= np.exp2(np.arange(M) % 41 - 20).astype(np.float32)[:, None]      # rows of very different size
        planes, xb, yb = gpu.planes(fmt, t), gpu.up(x), gpu.up(np.full(M * N, np.nan, np.float32))
        y = _call(gpu, fmt, xb, planes, yb, M, K, N, 0)
        again = _call(gpu, fmt, xb, planes, yb, M, K, N, 0)
        ref = _call(gpu, fmt, xb, planes, yb, M, K, N, 13)
        assert np.array_equal(y.view(np.uint32), ref.view(np.uint32))
        assert np.array_equal(again.view(np.uint32), ref.view(np.uint32))
        rows = [0, M // 2, M - 1] if N * K < 1 << 25 else [M - 1]
        order = {"q8": ("codes", "sc"), "q4": ("nib", "sc", "mn"), "q3": ("lo", "hi", "sc", "mn")}[fmt]
        r, den = getattr(O, "matmul_t_" + fmt)(np.ascontiguousarray(x[rows]), *[t[p] for p in order], len(rows), K, N,
                                               absden=True)
        assert np.all(np.abs(y[rows].astype(np.float64) - r) <= 1e-3 * den + 1e-30)
    finally:
        gpu.free()


def test_frag_non_finite(ctx):
    """An infinite and a NaN activation and a group of infinite scale stay where they belong, as in the tiled
    GEMM (a NaN is any NaN)."""
    M, K, N = 2048, 2080, 1000
    gpu = Gpu(ctx)
    try:
        t = synth.q4_tensor(3, N, K)
        t["sc"] = t["sc"].copy()
        t["sc"][7 * (K // 32) + 64] = 0x7C00          # the last group of column 7
        x = synth.normal(4, M * K).reshape(M, K)
        x[5, 3], x[2047, 2079], x[100] = np.inf, np.nan, 0.0
        planes, xb, yb = gpu.planes("q4", t), gpu.up(x), gpu.up(np.zeros(M * N, np.float32))
        y = _call(gpu, "q4", xb, planes, yb, M, K, N, 0)
        ref = _call(gpu, "q4", xb, planes, yb, M, K, N, 13)
        assert np.array_equal(np.isnan(y), np.isnan(ref))
        assert np.array_equal(np.where(np.isnan(y), 0, y), np.where(np.isnan(ref), 0, ref))
        assert not np.isfinite(y[5]).any() and np.isfinite(np.delete(y[6:2047], 7, 1)).all()
    finally:
        gpu.free()


def test_frag_workspaces_and_graphs():
    """A graph recorded of a smaller call stays valid across a call that takes the fragment GEMM with the same
    row staging, and such a call can itself be recorded (it then runs tiled, the same bits)."""
    M, K, N = 2045, 2560, 1024
    with Context(0) as ctx:
        gpu = Gpu(ctx)
        t = synth.q4_tensor(8, N, K)
        planes = gpu.planes("q4", t)
        xb = gpu.up(synth.normal(9, M * K))
        y1, y2, y3 = (gpu.up(np.zeros(M * N, np.float32)) for _ in range(3))
        small = 64
        ctx.matmul_t_q4(xb, *planes, y1, M, K, small)
        ref_small = ctx.download(y1, np.float32, M * small)
        ctx.graph_begin()
        ctx.matmul_t_q4(xb, *planes, y1, M, K, small)
        g1 = ctx.graph_end()
        ctx.matmul_t_q4(xb, *planes, y2, M, K, N)
        assert ctx.last_kernel() == "gemm_frag"
        ref = ctx.download(y2, np.float32, M * N)
        ctx.graph_begin()
        ctx.matmul_t_q4(xb, *planes, y3, M, K, N)
        assert ctx.last_kernel() == "gemm"
        g2 = ctx.graph_end()
        for _ in range(3):
            g1.launch()
            g2.launch()
            assert np.array_equal(ctx.download(y1, np.float32, M * small), ref_small)
            assert np.array_equal(ctx.download(y3, np.float32, M * N), ref)
            ctx.matmul_t_q4(xb, *planes, y2, M, K, N)
            assert np.array_equal(ctx.download(y2, np.float32, M * N), ref)
        g1.destroy()
        g2.destroy()
        gpu.free()


def test_frag_workspace_history():
    """Rows whose plain f16 form fits the workspace that fewer rows left, and whose whole panels of 32 would
    not: the call takes the fragment GEMM all the same, and a graph recorded before it stays valid."""
    K, N = 17024, 1000
    with Context(0) as ctx:
        gpu = Gpu(ctx)
        t = synth.q3_tensor(12, N, K)
        planes = gpu.planes("q3", t)
        x = synth.normal(13, 1025 * K)
        xb, yb = gpu.up(x), gpu.up(np.zeros(1025 * N, np.float32))
        _call(gpu, "q3", xb, planes, yb, 1015, K, N, 13)
        ctx.graph_begin()
        ctx.matmul_t_q3(xb, *planes, yb, 1025, K, N)
        g = ctx.graph_end()
        g.launch()
        ref = ctx.download(yb, np.float32, 1025 * N).reshape(1025, N)
        y = _call(gpu, "q3", xb, planes, yb, 1025, K, N, 0)
        assert np.array_equal(y.view(np.uint32), ref.view(np.uint32))
        g.launch()
        assert np.array_equal(ctx.download(yb, np.uint32, 1025 * N), ref.view(np.uint32).ravel())
        g.destroy()
        gpu.free()
