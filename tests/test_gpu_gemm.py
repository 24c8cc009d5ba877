"""The prompt GEMM (gemmDP4A, models/qwen3.js:1326-1407, more than 16 tokens) at the edges of its tiles: each f32 sum
of s_w * s_x * dot against 64 bits on the codes that quantQ8T gives, and the forward that is built on it."""
import numpy as np
import pytest

from tabinfer_amd import abi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = abi.Ctx(0)
    yield c
    c.close()


# K: one group, a remainder of the 4-group step, fewer steps than waves, whole rounds of them; N and T: one below,
# at and above a 16-wide tile; between them every tile shape of the dispatch at 256 CUs (the last five: 2 x 4 and
# 4 x 4 of 4 waves, 1 x 2, 1 x 4 and 2 x 3 of 8)
@pytest.mark.parametrize("T,N,K", [(2, 15, 32), (5, 17, 96), (16, 16, 160), (17, 33, 1120), (33, 4000, 288), (48, 4096, 64),
                                   (77, 2048, 2048), (95, 2064, 1056), (49, 4112, 320), (128, 4096, 128), (77, 6144, 96),
                                   (256, 100, 3104), (5, 8000, 2016), (200, 6000, 256), (255, 9999, 64), (31, 3000, 160),
                                   (128, 2048, 1120), (47, 6100, 96)])
def test_prompt_gemm_against_64_bits(ctx, orc, T, N, K):
    rng = np.random.default_rng(T * 7 + N + K)
    G = K // 32
    q = rng.integers(0, 16, (N, K), dtype=np.uint8)
    q[0] = 0                                        # a row of -8: with codes of +-127 the largest dots
    pack = (q[:, 0::2] | (q[:, 1::2] << 4)).copy()
    sc = rng.uniform(-0.03, 0.03, N * G).astype(np.float16)
    x = rng.standard_normal((T, K)).astype(np.float32)
    x[0, :32] = 0                                   # a group whose scale is 0
    x[-1] = np.where(rng.integers(0, 2, K), 3.0, -3.0)
    y0 = rng.standard_normal(T * N).astype(np.float32)
    dp, dx, dy = ctx.upload(pack), ctx.upload(x), ctx.upload(y0)
    dsc = ctx.upload(np.concatenate([np.zeros(1, np.float16), sc]))     # scales at an odd half-word
    ctx.call("ti_linear_q4", dx, dp, dsc.at(2), dy, T, N, K, 1)
    acc = ctx.download(dy, np.float32, T * N).reshape(T, N)
    ctx.call("ti_linear_q4", dx, dp, dsc.at(2), dy, T, N, K, 0)
    out = ctx.download(dy, np.float32, T * N).reshape(T, N)
    for b in (dp, dx, dy, dsc):
        b.free()
    xq, xs = orc.quant_act_q8_t(x.ravel(), T, K)
    codes = np.ascontiguousarray(xq).view(np.int8).reshape(T, G, 32).astype(np.float64)
    w = q.reshape(N, G, 32).astype(np.float64) - 8.0
    sw, sx = sc.reshape(N, G).astype(np.float64), np.asarray(xs, np.float64).reshape(T, G)
    for t in sorted({0, 1, T // 2, T - 1}):
        terms = np.einsum("ngk,gk->ng", w, codes[t]) * sw * sx[t]
        ref = terms.sum(1)
        # per group a rounded product of scales and an fma, then the sums of at most 8 waves
        tol = (G + 10) * 2.0 ** -24 * np.abs(terms).sum(1)
        assert np.all(np.abs(out[t] - ref) <= tol), t
        old = y0.reshape(T, N)[t].astype(np.float64)
        assert np.all(np.abs(acc[t] - (old + ref)) <= tol + 2.0 ** -23 * (np.abs(old) + np.abs(ref))), t


CFG = dict(layers=2, hidden=512, intermediate=1056, n_heads=4, n_kv_heads=2, head_dim=64, vocab=500, rope_theta=1e6, rms_eps=1e-6,
           max_ctx=300)


@pytest.mark.parametrize("T,pos", [(2, 0), (17, 5), (33, 0), (100, 64), (256, 0)])
def test_prompt_forward_is_its_short_chunks(ctx, T, pos):
    """A forward of T tokens against the same tokens one forward each (the GEMV kernels): logits, KV scales, next token."""
    rng = np.random.default_rng(T)
    shapes = {"self_attn.q_proj": (256, 512), "self_attn.k_proj": (128, 512), "self_attn.v_proj": (128, 512),
              "self_attn.o_proj": (512, 256), "mlp.gate_proj": (1056, 512), "mlp.up_proj": (1056, 512), "mlp.down_proj": (512, 1056)}
    w = {"model.embed_tokens.weight": (rng.standard_normal((500, 512)) * 0.5).astype(np.float16),
         "model.norm.weight": np.ones(512, np.float16)}
    lins = {"lm_head.weight": (500, 512)}
    for l in range(CFG["layers"]):
        lins.update({"model.layers.%d.%s.weight" % (l, n): s for n, s in shapes.items()})
        for n, k in (("input_layernorm", 512), ("post_attention_layernorm", 512), ("self_attn.q_norm", 64), ("self_attn.k_norm", 64)):
            w["model.layers.%d.%s.weight" % (l, n)] = (1 + 0.1 * rng.standard_normal(k)).astype(np.float16)
    packs = {n: (rng.integers(0, 256, a * b // 2, dtype=np.uint8), (rng.uniform(0.002, 0.01, a * b // 32)).astype(np.float16))
             for n, (a, b) in lins.items()}
    ids = rng.integers(0, 500, pos + T).astype(np.int32)
    res = []
    for chunk in (1, T):
        m = abi.Qwen3(ctx, max_tokens=256, **CFG)
        for n, v in w.items():
            ctx.write(m.tensor(n)[0], v)
        for n, (p, s) in packs.items():
            d, _, sd, _ = m.tensor(n)
            ctx.write(d, p)
            ctx.write(sd, s)
        if pos:
            m.forward(ids[:pos], 0) if chunk > 1 else [m.forward(ids[t:t + 1], t) for t in range(pos)]
        for t in range(0, T, chunk):
            m.forward(ids[pos + t:pos + t + chunk], pos + t)
        ks = [ctx.download(m.kv(l)[1], np.float32, (pos + T) * 2 * 2) for l in range(CFG["layers"])]
        res.append((ctx.download(m.logits_ptr(), np.float32, 500), ks, int(m.read_tokens(pos + T, 1)[0])))
        m.close()
    (a, ka, ta), (b, kb, tb) = res

    def rel(u, v):
        return np.linalg.norm(u - v) / np.linalg.norm(v)

    # The first layer's rows see the same codes but for those on a rounding boundary: one code of
    # K = 512 terms of rms 35 codes moves a projection by 1 / (35 sqrt(512)) = 1.3e-3 of its rms.
    assert rel(ka[0], kb[0]) < 1.4e-3
    # Behind it the codes of each of 4 quantized inputs a layer and of the cache rows may all round
    # otherwise: 0.289 codes of 35 rms (45 in the cache) on either side, sqrt(2 * 10) * 0.289 / 35.
    assert rel(ka[1], kb[1]) < 0.037 and rel(a, b) < 0.037
    assert tb == int(np.argmax(b)) and ta == int(np.argmax(a))
