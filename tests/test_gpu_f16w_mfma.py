"""The f16-weight product on the matrix cores: the few-row GEMM (2 to 64 rows) and the GEMM over x fragments
with W rows through LDS (gemm_frag.hip), each tile of both, against the oracle at the matmul bar (1e-3 of
sum |x w|). K ends at every remainder of 32 that the entry point takes there (multiples of 8), so the last
step's chunks past K, which hold the next row's values, have to count as zeros: an infinite weight at the
start of a row must not reach the row before it.
"""
import numpy as np
import pytest

import oracle as O
from brimkern_amd.capi import BRIK_OPT_SPLITK, Context
from helpers import Gpu

pytestmark = pytest.mark.gpu


@pytest.fixture()
def gpu(ctx):
    g = Gpu(ctx)
    yield g
    ctx.set_option(BRIK_OPT_SPLITK, 0)
    g.free()


def data(M, K, N, seed):
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal((M, K)) * np.exp2(np.arange(M) % 37 - 18)[:, None]).astype(np.float32)
    return x, (rng.standard_normal((N, K)) * 0.05).astype(np.float16)


def run(gpu, x, w):
    (M, K), N = x.shape, w.shape[0]
    yb = gpu.up(np.full(M * N, np.nan, np.float32))
    gpu.ctx.matmul_t_f16w(gpu.up(x), gpu.up(w.view(np.uint16)), yb, M, K, N)
    return gpu.ctx.download(yb, np.float32, M * N).reshape(M, N)


def check(y, x, w):
    ref, den = O.matmul_t_f16w(x.ravel(), w.view(np.uint16).ravel(), *x.shape, w.shape[0])
    assert np.all(np.abs(y - ref) <= 1e-3 * den + 1e-30)


@pytest.mark.parametrize("M,K,N", [
    (4096, 288, 2560), (4095, 72, 2555),      # 192 x 256
    (512, 520, 9728), (500, 64, 9701),        # 256 x 128
    (777, 1000, 4096), (770, 32, 4090),       # 128 x 128
    (130, 40, 333), (65, 8, 70), (200, 1048, 129), (100, 10248, 65),   # 64 x 64; one chunk of K; rows read twice
])
def test_h_tiles(gpu, M, K, N):
    x, w = data(M, K, N, M + K)
    y = run(gpu, x, w)
    assert gpu.ctx.last_kernel() == "gemm_h"
    check(y, x, w)
    assert np.array_equal(y.view(np.uint32), run(gpu, x, w).view(np.uint32))


@pytest.mark.parametrize("M,K,N", [(2, 8, 33), (8, 1032, 127), (9, 264, 129), (16, 2568, 200), (17, 40, 130),
                                   (32, 1304, 257), (24, 5152, 65), (33, 24, 513), (64, 544, 127), (47, 3104, 130)])
def test_few_f16(gpu, M, K, N):
    x, w = data(M, K, N, M + K + 1)
    gpu.ctx.set_option(BRIK_OPT_SPLITK, 3)
    check(run(gpu, x, w), x, w)
    assert gpu.ctx.last_kernel() == "gemm_few"


@pytest.mark.parametrize("M,kernel", [(5, "gemm_few"), (40, "gemm_few"), (40, "gemm_h"), (200, "gemm_h")])
@pytest.mark.parametrize("K", [40, 64, 72, 88])
def test_infinite_weight_stays_in_its_row(gpu, M, K, kernel):
    N = 70
    gpu.ctx.set_option(BRIK_OPT_SPLITK, 3 if kernel == "gemm_few" else 1)
    x, w = data(M, K, N, 7)
    x = np.abs(x) + np.float32(0.5)
    w[7, 0] = w[69, K - 1] = np.float16(np.inf)
    y = run(gpu, x, w)
    assert gpu.ctx.last_kernel() == kernel
    cols = [n for n in range(N) if n not in (7, 69)]
    assert np.isposinf(y[:, [7, 69]]).all() and np.isfinite(y[:, cols]).all()
    check(y[:, cols], x, np.ascontiguousarray(w[cols]))


@pytest.mark.parametrize("M,K", [(40, 40), (100, 40), (100, 72), (300, 88), (2000, 72)])
def test_weights_that_end_their_allocation(gpu, M, K):
    """W of whole 64 KiB in an allocation of its own: the last row's last step has 8, 16 or 24 of 32 k inside."""
    N = 4096
    assert N * K * 2 % 65536 == 0
    x, w = data(M, K, N, M * K)
    gpu.ctx.set_option(BRIK_OPT_SPLITK, 1)
    check(run(gpu, x, w), x, w)
    assert gpu.ctx.last_kernel() == "gemm_h"


@pytest.mark.parametrize("K", [9728, 9736])
def test_workspace_history(K):
    """97 rows fit, as plain f16 rows, the workspace that 80 rows leave; whole panels of 32 do not. Such a call
    runs the same kernel as after a larger one, and recorded there (the workspace may not grow, an older kernel
    stands in) it gives the same bits."""
    N = 96
    x, w = data(400, K, N, 11)
    with Context(0) as c:
        gpu = Gpu(c)
        xb, wb, yb = gpu.up(x), gpu.up(w.view(np.uint16)), gpu.up(np.zeros(400 * N, np.float32))

        def call(M):
            c.matmul_t_f16w(xb, wb, yb, M, K, N)
            return c.last_kernel()

        def result():
            r = c.download(yb, np.uint32, 97 * N)
            c.h2d(yb, np.zeros(97 * N, np.float32))
            return r

        assert call(80) == "gemm_h"
        c.graph_begin()
        assert call(97) != "gemm_h"
        g = c.graph_end()
        g.launch()
        recorded = result()
        assert call(97) == "gemm_h"
        first = result()
        g.launch()                       # the call before left the workspace where it was
        assert np.array_equal(result(), recorded) and np.array_equal(first, recorded)
        g.destroy()
        assert call(400) == "gemm_h" and call(97) == "gemm_h"
        assert np.array_equal(result(), first)
        check(first.view(np.float32).reshape(97, N), x[:97], w)
        gpu.free()
