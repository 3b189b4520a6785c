"""The few-row GEMM (gemm_few.hip, 2 to 64 rows, x staged in the launch), forced through the few-row option,
against the oracle: every tile (rows 8 / 16 / 32 / 64), piece counts on both sides of one per k wave, K ends
inside a piece and inside a step, ragged columns, one and several K slices.

Bar: f16 operands (x and W rounded to 11 bits, 2^-11 each at most) with f32 sums stay within 2^-10 of
sum |x w| plus the f32 sums' part, under 1e-3.
"""
import numpy as np
import pytest

import oracle as O
from brimkern_amd import synth
from brimkern_amd.capi import BRIK_OPT_PATH, BRIK_OPT_SPLITK, BRIK_PATH_SPLITK
from helpers import Gpu, PLANES, REL_TOL

pytestmark = pytest.mark.gpu


@pytest.fixture()
def gpu(ctx):
    g = Gpu(ctx)
    ctx.set_option(BRIK_OPT_SPLITK, 3)
    ctx.set_option(BRIK_OPT_PATH, 2)
    yield g
    ctx.set_option(BRIK_OPT_SPLITK, 0)
    ctx.set_option(BRIK_OPT_PATH, 0)
    g.free()


def run(gpu, fmt, t, x, M):
    y = gpu.matmul(fmt, x, gpu.planes(fmt, t), M, t["K"], t["N"])
    assert gpu.ctx.last_path() == BRIK_PATH_SPLITK and gpu.ctx.last_kernel() == "gemm_few"
    r, den = getattr(O, f"matmul_t_{fmt}")(x, *[t[k] for k in PLANES[fmt]], M, t["K"], t["N"], absden=True)
    return y, r, den


@pytest.mark.parametrize("fmt", ["q4", "q8", "q3"])
@pytest.mark.parametrize("M,K,N", [
    (2, 256, 33), (7, 288, 600), (8, 1056, 127),          # 8 rows
    (9, 224, 129), (16, 1024, 31),                        # 16 rows, at most 4 pieces
    (9, 1056, 777), (16, 2560, 200),                      # 16 rows, more
    (17, 96, 130), (32, 1312, 257), (24, 5152, 65),       # 32 rows; 21 pieces in several slices
    (33, 32, 513), (64, 544, 127), (47, 3104, 130),       # 64 rows; one group of K
])
def test_few_shapes(gpu, fmt, M, K, N):
    t = synth.tensor(fmt, 2000 + M + K, N, K)
    x = synth.normal(2001 + M, M * K)
    y, r, den = run(gpu, fmt, t, x, M)
    assert np.all(np.abs(y.astype(np.float64) - r) <= REL_TOL * den + 1e-30)


@pytest.mark.parametrize("M,K,N", [(8, 1056, 130), (16, 1056, 130), (32, 1056, 130), (64, 1056, 130)])
def test_few_pieces_of_any_size(gpu, M, K, N):
    """Rows whose 256-wide pieces differ by forty orders of magnitude, a zero row, and rows with an infinity or
    a NaN in one piece: each piece takes its own scale, and only the rows concerned stop being finite."""
    t = synth.q4_tensor(2100, N, K)
    x = synth.normal(2101, M * K).reshape(M, K)
    for i in range(0, K, 256):
        x[:, i:i + 256] *= np.float32(10.0) ** ((i // 256 * 13) % 41 - 20)
    x[1] = 0
    y, r, den = run(gpu, "q4", t, x, M)
    assert np.all(np.abs(y.astype(np.float64) - r) <= REL_TOL * den + 1e-30) and not y[1].any()
    x[3, 300], x[M - 1, K - 1] = np.inf, np.nan
    y2 = gpu.matmul("q4", x, gpu.planes("q4", t), M, K, N)
    fine = [m for m in range(M) if m not in (3, M - 1)]
    assert np.array_equal(y2[fine], y[fine])
    assert not np.isfinite(y2[3]).any() and np.isnan(y2[M - 1]).all()


def test_few_last_rows_and_scales(gpu):
    """Weights whose last column's scales end the plane inside a 16-byte load, at every remainder of the group
    count mod 8, and a matrix of 16 groups in all."""
    for K, N in [(32, 16), (64, 9), (96, 7), (288, 3), (320, 5), (352, 3), (416, 3), (480, 2), (512, 1)]:
        t = synth.q3_tensor(2200 + K, N, K)
        x = synth.normal(2201 + K, 5 * K)
        y, r, den = run(gpu, "q3", t, x, 5)
        assert np.all(np.abs(y.astype(np.float64) - r) <= REL_TOL * den + 1e-30), (K, N)


# wide matrices of 33 rows or more, which the model of the split-K kernel would take, and one whose best slice count
# would not fit the no-allocation scratch (fewer slices do)
@pytest.mark.parametrize("fmt,M,K,N", [("q4", 36, 3200, 9728), ("q8", 40, 3200, 12000), ("q3", 64, 4096, 9728),
                                       ("q4", 64, 9728, 8192)])
def test_few_in_place_of_splitk(gpu, fmt, M, K, N):
    gpu.ctx.set_option(BRIK_OPT_SPLITK, 0)
    gpu.ctx.set_option(BRIK_OPT_PATH, 0)
    t = synth.tensor(fmt, 2300 + M, N, K)
    x = synth.normal(2301 + M, M * K)
    y = gpu.matmul(fmt, x, gpu.planes(fmt, t), M, K, N)
    assert gpu.ctx.last_kernel() == "gemm_few"
    deq = getattr(O, f"dequant_{fmt}")(*[t[k] for k in PLANES[fmt]]).reshape(N, K)
    cols = np.r_[0:40, N - 40:N]
    w, xd = deq[cols].astype(np.float64).T, x.reshape(M, K).astype(np.float64)
    assert np.all(np.abs(y[:, cols] - xd @ w) <= REL_TOL * (np.abs(xd) @ np.abs(w)))
