"""The matrix-core int3 expert GEMM (moeSort + moeGemm3, models/lfm25.js:1503-1647) at the edges of its tiles: each f32 sum
of s_w * s_x * dot against 64 bits on the codes that quantAct8 gives."""
import numpy as np
import pytest

from tabinfer_amd import abi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = abi.Ctx(0)
    yield c
    c.close()


# K: one group, a remainder of the 4-group step, whole rounds of the waves' steps; N around a 16- and a 64-row tile;
# counts: pairs per expert (five or more on average), around the 16-pair tile, the 32-pair pass and the 1024-pair scan, and none
@pytest.mark.parametrize("N,K,counts,div", [(15, 32, (1, 0, 15), 1), (17, 160, (16, 17), 2), (64, 2048, (33, 3, 0, 1), 4),
                                            (65, 4096, (2, 32), 1), (100, 2080, (700, 5, 570), 5), (48, 544, (0, 0, 37, 0, 2, 1, 0, 0), 1)])
def test_moe_gemm_against_64_bits(ctx, orc, N, K, counts, div):
    rng = np.random.default_rng(N + K)
    nE, G, P = len(counts), K // 32, sum(counts)
    q = rng.integers(0, 8, (nE * N, G, 32), dtype=np.uint8)
    q[0] = 0                                        # a row of -4
    planes = np.stack([np.packbits((q >> b) & 1, axis=-1, bitorder="little") for b in range(3)], 2)
    sc = rng.uniform(-0.03, 0.03, (nE * N, G)).astype(np.float16)
    ridx = rng.permutation(np.repeat(np.arange(nE), counts)).astype(np.int32)
    rows = (P - 1) // div + 1
    x = rng.standard_normal((rows, K)).astype(np.float32)
    x[0, :32] = 0                                   # a group whose scale is 0
    x[-1] = np.where(rng.integers(0, 2, K), 3.0, -3.0)
    bufs = [ctx.upload(a) for a in (x, planes, sc, ridx)]
    dy = ctx.upload(np.full(P * N, np.nan, np.float32))
    ctx.call("ti_moe_gemm_q3", bufs[0], rows, *bufs[1:], dy, P, N, K, div, nE)
    out = ctx.download(dy, np.float32, P * N).reshape(P, N)
    for b in bufs + [dy]:
        b.free()
    xq, xs = orc.quant_act_q8_t(x.ravel(), rows, K)
    codes = np.ascontiguousarray(xq).view(np.int8).reshape(rows, G, 32).astype(np.float64)
    sx = np.asarray(xs, np.float64).reshape(rows, G)
    for p in sorted({0, P // 3, P // 2, P - 1}):
        e, t = ridx[p], p // div
        w = q[e * N:(e + 1) * N].astype(np.float64) - 4.0
        terms = np.einsum("ngk,gk->ng", w, codes[t]) * sc[e * N:(e + 1) * N].astype(np.float64) * sx[t]
        # per group a rounded product of scales and an fma, then the sums of four waves
        assert np.all(np.abs(out[p] - terms.sum(1)) <= (G + 6) * 2.0 ** -24 * np.abs(terms).sum(1)), p
    assert not np.isnan(out).any()
