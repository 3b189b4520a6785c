"""The softcap / penalty pass at the edges of its blocks (1024 logits) and of its threads (4 logits), the
vector at every 4-byte alignment, recent ids on both sides of each edge.

Logits are evenly spaced and shuffled, so no rounding changes a rank. Tolerance of the values: tanhf (5 ulp, 10 roundings of 2^-24),
the division and product of the softcap and the penalty's division or product: under 16 roundings of 2^-24 on each side.
"""
import numpy as np
import pytest

from helpers import Gpu
from test_gpu_topk import oracle_passes

pytestmark = pytest.mark.gpu


@pytest.fixture()
def gpu(ctx):
    g = Gpu(ctx)
    yield g
    g.free()


@pytest.mark.parametrize("offset", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [3, 4, 5, 1023, 1024, 1025, 2047, 4098])
def test_topk_prep_edges(gpu, n, offset):
    rng = np.random.default_rng(n)
    logits = rng.permutation(np.linspace(-9, 9.1, n).astype(np.float32))
    recent = sorted({i for i in (0, 1, 3, 4, 1022, 1023, 1024, 2046, 2047, 2048, n - 1) if i < n})
    k = min(n, 64)
    guard = np.full(8, 77.0, np.float32)
    lb = gpu.up(np.concatenate([guard[:4 + offset], logits, guard]))
    rb = gpu.up(np.asarray(recent, np.int32))
    ob = gpu.up(np.zeros(2 * k, np.int32))
    gpu.ctx.logits_topk(lb.offset(4 * (4 + offset)), n, rb, len(recent), 1.25, 30.0, k, ob, ob.offset(4 * k))
    ids, vals = gpu.ctx.download(ob, np.int32, k), gpu.ctx.download(ob, np.float32, k, src_offset=4 * k)
    after = gpu.ctx.download(lb, np.float32, n + 12 + offset)
    ref, rids, rvals = oracle_passes(logits, recent, 1.25, 30.0, k)
    tol = 2.0 ** -19
    np.testing.assert_allclose(after[4 + offset:4 + offset + n], ref, rtol=tol, atol=tol)
    assert np.all(after[:4 + offset] == 77) and np.all(after[4 + offset + n:] == 77)
    np.testing.assert_allclose(vals, rvals, rtol=tol, atol=tol)
    np.testing.assert_allclose(ref[ids], rvals, rtol=tol, atol=tol)
    assert len(set(ids.tolist())) == k
