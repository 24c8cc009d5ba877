"""The prompt attention kernel (attnBlock's T > 1 case, models/qwen3.js:2534-2577) at the edges of its row tiles, key blocks
and key ranges, against softmax attention in 64 bits."""
import numpy as np
import pytest

from tabinfer_amd import abi

pytestmark = pytest.mark.gpu
HD = 128


@pytest.fixture(scope="module")
def ctx():
    c = abi.Ctx(0)
    yield c
    c.close()


# T x heads per KV head: one above the short kernel's 32 rows, around 64 and 128 rows, several workgroups; contexts from
# the chunk alone to several ranges with a remainder, and past 16384 keys, where 64 ranges grow. wide: V scales over six decades, a V above the f16 range
@pytest.mark.parametrize("T,pos,nHq,nKv,wide", [(33, 0, 2, 2, False), (17, 62, 4, 2, True), (32, 64, 4, 2, False), (33, 31, 4, 2, True),
                                                (65, 127, 2, 1, False), (11, 100, 12, 4, False), (64, 1000, 16, 4, True),
                                                (256, 0, 2, 1, False), (100, 2777, 16, 8, True), (256, 1100, 8, 8, False),
                                                (33, 17001, 2, 2, False)])
def test_prompt_attention_against_64_bits(ctx, T, pos, nHq, nKv, wide):
    rng = np.random.default_rng(T + pos + nHq)
    S = pos + T
    q = (rng.standard_normal((T, nHq, HD)) * rng.choice([0.3, 3.0], (T, nHq, 1))).astype(np.float32)
    kc, vc = (rng.integers(-127, 128, (S, nKv, HD)).astype(np.int8) for _ in range(2))
    ks, vs = (rng.uniform(0.5, 3.0, (S, nKv, HD // 32)).astype(np.float32) for _ in range(2))
    if wide:
        vs *= (10.0 ** rng.uniform(-3, 3, vs.shape)).astype(np.float32)
        vs[S // 2] = 1e5
    check(ctx, q, kc, ks, vc, vs, pos)


def check(ctx, q, kc, ks, vc, vs, pos):
    (T, nHq, _), (S, nKv) = q.shape, kc.shape[:2]
    G = nHq // nKv
    bufs = [ctx.upload(a) for a in (q, kc, ks, vc, vs)] + [ctx.upload(np.full(T * nHq * HD, np.nan, np.float32))]
    ctx.call("ti_attn_causal_q8", *bufs, T, pos, nHq, nKv, HD)
    out = ctx.download(bufs[-1], np.float32, T * nHq * HD).reshape(T, nHq, HD)
    for b in bufs:
        b.free()
    K = kc.astype(np.float64) * np.repeat(ks.astype(np.float64) / 127, 32, -1)
    V = vc.astype(np.float64) * np.repeat(vs.astype(np.float64) / 127, 32, -1)
    seen = np.arange(S)[None] <= pos + np.arange(T)[:, None]
    for h in range(nHq):
        k, v, x = K[:, h // G], V[:, h // G], q[:, h].astype(np.float64)
        s = np.where(seen, x @ k.T / np.sqrt(HD), -np.inf)
        p = np.exp(s - s.max(-1, keepdims=True))
        p /= p.sum(-1, keepdims=True)
        # a score is off by the split of q and four rounded group sums, at most 2^-21 of sum |q k|, on either side of
        # the softmax; a weight by the exponential and its product with the V scale (2^-20), whatever the scales of
        # the other keys; the sums of S terms by S / 2^24
        ds = 2 * 2.0 ** -21 * np.where(seen, np.abs(x) @ np.abs(k).T / np.sqrt(HD), 0).max(-1)
        tol = (ds[:, None] + 2.0 ** -20 + 2 * S * 2.0 ** -24) * (p @ np.abs(v))
        assert np.all(np.abs(out[:, h] - p @ v) <= tol), h


# Each row's weights keep f32 accuracy beside a V scale 2^up as large: that of a token the row does not see, or
# (seen) of keys that it gives next to no weight, one in each block of 64
@pytest.mark.parametrize("up", [12, 20, 30, 60])
@pytest.mark.parametrize("seen", [False, True])
def test_prompt_attention_beside_large_v_scales(ctx, up, seen):
    rng = np.random.default_rng(up)
    T, pos, nHq, nKv = 80, 300, 4, 2
    S = T + pos
    q = rng.standard_normal((T, nHq, HD)).astype(np.float32)
    kc, vc = (rng.integers(-127, 128, (S, nKv, HD)).astype(np.int8) for _ in range(2))
    ks, vs = (rng.uniform(0.5, 1.5, (S, nKv, HD // 32)).astype(np.float32) for _ in range(2))
    if seen:                                        # a score of 0.28 against -35 - 0.69 up: the weight falls as the scale grows
        q[..., 0] = 20.0
        kc[..., 0] = 20
        ks[..., 0] = 1.0
        kc[5::64, :, 0] = -127
        ks[5::64, :, 0] = (35.0 + 0.7 * up) * np.sqrt(HD) / 20.0
        vs[5::64] *= np.float32(2.0 ** up)
    else:
        vs[-1] *= np.float32(2.0 ** up)
    check(ctx, q, kc, ks, vc, vs, pos)
