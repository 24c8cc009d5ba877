"""The attention of a T = 2..16 token forward (attnBlock's T > 1 case, models/qwen3.js:2534-2577) against softmax attention
in 64 bits: the forward's trace holds the scale of every 32 outputs, their largest / 127 in f32."""
import numpy as np
import pytest

from tabinfer_amd import abi
import qwen3_tf as TF

pytestmark = pytest.mark.gpu

CFG = dict(layers=1, hidden=256, intermediate=512, n_heads=16, n_kv_heads=8, head_dim=128, vocab=1000, rope_theta=1e6,
           rms_eps=1e-6, max_ctx=64, max_tokens=16)
P, T, HD = 24, 16, 128


@pytest.fixture(scope="module")
def ctx():
    c = abi.Ctx(0)
    yield c
    c.close()


def heads64(x, w, pos0):
    """RMSNorm and rotary embedding of x [T][heads][128] in 64 bits."""
    x = x.astype(np.float64)
    x = x / np.sqrt((x * x).mean(-1, keepdims=True) + CFG["rms_eps"]) * w.view(np.float16).astype(np.float64)
    a = (pos0 + np.arange(len(x)))[:, None, None] * CFG["rope_theta"] ** (-2.0 * np.arange(64) / HD)
    lo, hi = x[..., :64], x[..., 64:]
    return np.concatenate([lo * np.cos(a) - hi * np.sin(a), hi * np.cos(a) + lo * np.sin(a)], -1)


# Sharp softmaxes (a few keys share each row) over 8192 rows, so that weights on a rounding boundary of their
# 16-bit parts are among them; up: the V scales of the cache, which the outputs follow
@pytest.mark.parametrize("up", [0, -18, 14])
def test_short_batch_attention_against_64_bits(ctx, up):
    rng = np.random.default_rng(3)
    W = TF.make_weights(CFG, 3, range(CFG["vocab"]))
    p = "model.layers.0.self_attn."
    W[p + "q_norm.weight"] = np.full(HD, 4.0, np.float16).view(np.uint16)
    w, sw = W[p + "v_proj.weight"]                  # the new keys' V as the cache's
    W[p + "v_proj.weight"] = (w, (sw.view(np.float16) * np.float32(2.0 ** min(up, 0))).astype(np.float16).view(np.uint16))
    nH, nK = CFG["n_heads"], CFG["n_kv_heads"]
    m = abi.Qwen3(ctx, **CFG)
    worst = 0.0
    try:
        TF.load_into(ctx, m, W, CFG["hidden"])
        for rep in range(32):
            kv = TF.seed_prefix(ctx, m, CFG, P, CFG["max_ctx"], 100 + rep)[0]
            kv[3][:P * nK * 4] *= np.float32(2.0 ** up)
            ctx.write(m.kv(0)[3], kv[3][:P * nK * 4])
            layers, _ = TF.traced(ctx, m, CFG, lambda: m.forward(rng.integers(0, CFG["vocab"], T).astype(np.int32), P))
            new = TF.new_kv_rows(ctx, m, CFG, P, T)[0]
            K, V = [(np.concatenate([c.view(np.int8)[:P * nK * HD].reshape(P, -1), n.view(np.int8).reshape(T, -1)]).astype(np.float64)
                     * np.repeat(np.concatenate([s[:P * nK * 4].reshape(P, -1), ns]).astype(np.float64) / 127, 32, -1)).reshape(P + T, nK, HD)
                    for c, s, n, ns in ((kv[0], kv[1], new[0], new[1]), (kv[2], kv[3], new[2], new[3]))]
            q = heads64(layers[0]["q"][:T].reshape(T, nH, HD), W[p + "q_norm.weight"], P)
            got = 127.0 * layers[0]["a_s"][:T].astype(np.float64).reshape(T, nH, HD // 32)
            seen = np.arange(P + T)[None] <= P + np.arange(T)[:, None]
            for h in range(nH):
                k, v = K[:, h // 2], V[:, h // 2]
                s = np.where(seen, q[:, h] @ k.T / np.sqrt(HD), -np.inf)
                e = np.exp(s - s.max(-1, keepdims=True))
                e /= e.sum(-1, keepdims=True)
                # a score: the norm, rotation and split of q and four group sums, 2^-21 of sum |q k| on either side of the
                # softmax; a weight 2^-20; the sums 2 S / 2^24
                ds = 2 * 2.0 ** -21 * np.where(seen, np.abs(q[:, h]) @ np.abs(k).T / np.sqrt(HD), 0).max(-1)
                grp = lambda x: np.abs(x).reshape(T, 4, 32).max(-1)  # noqa: E731
                tol = (ds[:, None] + 2.0 ** -20 + 2 * (P + T) * 2.0 ** -24) * grp(e @ np.abs(v))
                worst = max(worst, float((np.abs(got[:, h] - grp(e @ v)) / tol).max()))
    finally:
        m.close()
    assert worst <= 1.0, worst
