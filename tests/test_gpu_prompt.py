"""Prompt forwards (T > 16 tokens of the Qwen3 stack, T >= 2 of the Bonsai stack; no trace: these kernels run without one)
against the same layers in 64 bits with the formats' own quantizers, token by token: the second layer's K and V rows,
which all of the first layer's kernels have gone into, and the logits. The attention of the 64-bit layers reads the
GPU's own cache rows, so a token's row depends on that token's int8 codes alone: it agrees to f32 rounding unless one
of them stood at a rounding boundary and was taken otherwise."""
import numpy as np
import pytest

from tabinfer_amd import abi
import bonsai_ref as B
import qwen3_tf as TF

pytestmark = pytest.mark.gpu
HD, EPS, THETA = 128, 1e-6, 1e6


@pytest.fixture(scope="module")
def ctx():
    c = abi.Ctx(0)
    yield c
    c.close()


def rms(x, w):
    return x / np.sqrt((x * x).mean(-1, keepdims=True) + EPS) * w


def rope(x, pos, angle=np.float64):
    i = np.arange(HD // 2)
    a = ((pos + np.arange(len(x)))[:, None].astype(angle) * (THETA ** (-2.0 * i / HD)).astype(angle))[:, None].astype(np.float64)
    lo, hi = x[..., :64], x[..., 64:]
    return np.concatenate([lo * np.cos(a) - hi * np.sin(a), hi * np.cos(a) + lo * np.sin(a)], -1)


def attend(q, k, v, pos):
    """q [T][heads][128] at pos.. over k, v [pos + T][KV heads][128], causal."""
    T, S, g = len(q), len(k), q.shape[1] // k.shape[1]
    seen = np.arange(S)[None] <= pos + np.arange(T)[:, None]
    out = np.empty_like(q)
    for h in range(q.shape[1]):
        s = np.where(seen, q[:, h] @ k[:, h // g].T / np.sqrt(HD), -np.inf)
        p = np.exp(s - s.max(-1, keepdims=True))
        out[:, h] = p @ v[:, h // g] / p.sum(-1, keepdims=True)
    return out


def silu_mul(g, u):
    return g / (1.0 + np.exp(-g)) * u


def check(got, want, logits, ref):
    """Rows [layer][K, V][T][..] and logits."""
    for l in range(2):
        for g, w in zip(got[l], want[l]):
            w = w.reshape(len(w), -1)
            e = np.linalg.norm(g.reshape(w.shape).astype(np.float64) - w, axis=1) / np.linalg.norm(w, axis=1)
            # f32 rounding, but for tokens with a code on its boundary: of a token's some 7 000 codes (rms 35, off by
            # 3e-7 of it) one in 10^5 each, and what follows from it
            assert (e > 2.0 ** -20).sum() <= max(1, 0.2 * len(e)), (l, np.sort(e))
            # one code is 1 / (35 sqrt(1024)) = 9e-4 of a projection; it may move some of the layer's others
            assert e.max() < 0.05, (l, np.sort(e))
    assert np.linalg.norm(logits - ref) < 0.05 * np.linalg.norm(ref)


# ---- Qwen3 --------------------------------------------------------------------------------------
def q8(x):
    v = x.astype(np.float32).reshape(-1, 32)
    s = np.abs(v).max(-1, keepdims=True) / np.float32(127)
    with np.errstate(divide="ignore"):
        inv = np.where(s > 0, np.float32(1) / s, np.float32(0))
    return (np.clip(np.rint(v * inv), -127, 127).astype(np.float64) * s).reshape(x.shape)


def int4_f64(val, N, K):
    p, s = val
    b = p.view(np.uint8)
    q = np.stack([b & 15, b >> 4], -1).reshape(N, K // 32, 32).astype(np.float64) - 8.0
    return (q * s.view(np.float16).astype(np.float64).reshape(N, K // 32, 1)).reshape(N, K)


def qwen_f64(cfg, W, kv, got, ids, P):
    d, T = TF.dims(cfg), len(ids)
    f16 = lambda n: W[n].view(np.float16).astype(np.float64)  # noqa: E731
    lin = lambda n, a: a @ int4_f64(W[n], *(d[k] for k in TF.SHAPES[n.split(".", 3)[3]])).T  # noqa: E731
    x = np.stack([W["emb_rows"][int(i)].view(np.float16).astype(np.float64) for i in ids])
    rows = []
    for l in range(cfg["layers"]):
        p = "model.layers.%d." % l
        a = q8(rms(x, f16(p + "input_layernorm.weight")))
        q, k, v = [lin(p + "self_attn.%s_proj.weight" % n, a).reshape(T, -1, HD) for n in "qkv"]
        q, k = [rope(rms(t, f16(p + "self_attn.%s_norm.weight" % n)), P) for t, n in ((q, "q"), (k, "k"))]
        rows.append([np.abs(t.reshape(T, -1, 32)).max(-1) for t in (k, v)])
        keys, vals = [(np.concatenate([c.view(np.int8)[:P * d["nkv"]], nc.view(np.int8).ravel()]).reshape(P + T, -1, 4, 32)
                       * (np.concatenate([s[:P * d["nkv"] // 32], ns.ravel()]).astype(np.float64) / 127).reshape(P + T, -1, 4, 1)
                       ).reshape(P + T, -1, HD) for c, s, nc, ns in (kv[l][:2] + got[l][:2], kv[l][2:] + got[l][2:])]
        o = attend(q, keys, vals, P).reshape(T, -1)
        x = x + lin(p + "self_attn.o_proj.weight", q8(o))
        a = q8(rms(x, f16(p + "post_attention_layernorm.weight")))
        x = x + lin(p + "mlp.down_proj.weight", q8(silu_mul(lin(p + "mlp.gate_proj.weight", a), lin(p + "mlp.up_proj.weight", a))))
    return rows, int4_f64(W["lm_head.weight"], cfg["vocab"], d["H"]) @ rms(x[-1], f16("model.norm.weight"))


# With 256 CUs the gate/up tile is 2, 4, 2 and 4 token tiles of 8 waves and 4 of 4 waves; the norm is run at and off the
# widths its instances end at; the attention runs one and several key ranges, with and without a prefix
@pytest.mark.parametrize("H,I,T,P", [(1024, 3072, 33, 5), (1024, 3072, 100, 0), (2048, 6144, 17, 70), (2048, 6144, 64, 0),
                                     (2048, 6144, 256, 130), (512, 1056, 40, 700), (256, 512, 20, 9), (3072, 512, 33, 0), (6144, 512, 18, 0)])
def test_prompt_layer_against_64_bits(ctx, H, I, T, P):
    cfg = dict(layers=2, hidden=H, intermediate=I, n_heads=16, n_kv_heads=8, head_dim=HD, vocab=512, rope_theta=THETA,
               rms_eps=EPS, max_ctx=P + T, max_tokens=T)
    W = TF.make_weights(cfg, H + T, range(cfg["vocab"]))
    for l in range(2):                              # few keys share a softmax, so a wrong one shows
        W["model.layers.%d.self_attn.q_norm.weight" % l] = np.full(HD, 3.0, np.float16).view(np.uint16)
    ids = np.random.default_rng(T).integers(0, cfg["vocab"], T).astype(np.int32)
    m = abi.Qwen3(ctx, **cfg)
    try:
        TF.load_into(ctx, m, W, H)
        kv = TF.seed_prefix(ctx, m, cfg, P, P + T, 4)
        m.forward(ids, P)
        got = TF.new_kv_rows(ctx, m, cfg, P, T)
        logits = ctx.download(m.logits_ptr(), np.float32, cfg["vocab"]).astype(np.float64)
    finally:
        m.close()
    rows, want = qwen_f64(cfg, W, [list(t) for t in kv], [list(t) for t in got], ids, P)
    check([(r[1], r[3]) for r in got], rows, logits, want)


# ---- Bonsai -------------------------------------------------------------------------------------
def n2(x):
    v = x.astype(np.float32)
    s = np.float32(127) / np.abs(v).max(-1, keepdims=True)
    y = v * s
    return np.clip(np.sign(y) * np.floor(np.abs(y) + np.float32(0.5)), -127, 127).astype(np.float64), s.astype(np.float64)


def tern_f64(val, N, K):
    b, s = val
    b = b.reshape(N, K // 64, 16)
    c = np.stack([b & 3, (b >> 2) & 3, (b >> 4) & 3, b >> 6], 2).reshape(N, K // 64, 64).astype(np.float64) - 1.0
    return (c * s.astype(np.float64).reshape(N, K // 64, 1)).reshape(N, K)


def bonsai_f64(cfg, W, pre, got, ids, P):
    d, T = B.dims(cfg), len(ids)

    def lin(n, a):
        return a[0] @ tern_f64(W[n], *(d[k] for k in B.SHAPES[n.split(".", 3)[3]])).T / a[1]
    x = np.stack([B.emb_row(W, i, d["H"]).view(np.float16).astype(np.float64) for i in ids])
    rows = []
    for l in range(cfg["layers"]):
        p = "model.layers.%d." % l
        a = n2(rms(x, W[p + "input_layernorm.weight"]))
        q, k, v = [lin(p + "self_attn.%s_proj.weight" % n, a).reshape(T, -1, HD) for n in "qkv"]
        q, k = [rope(rms(t, W[p + "self_attn.%s_norm.weight" % n]), P, np.float32) for t, n in ((q, "q"), (k, "k"))]   # the model's angles
        rows.append((k, v))
        o = attend(q, *[np.concatenate([pre[l][i], got[l][i]]).reshape(P + T, -1, HD).astype(np.float64) for i in range(2)], P)
        x = x + lin(p + "self_attn.o_proj.weight", n2(o.reshape(T, -1)))
        a = n2(rms(x, W[p + "post_attention_layernorm.weight"]))
        x = x + lin(p + "mlp.down_proj.weight", n2(silu_mul(lin(p + "mlp.gate_proj.weight", a), lin(p + "mlp.up_proj.weight", a))))
    a = n2(rms(x[-1:], W["model.norm.weight"]))
    return rows, (a[0] @ tern_f64(W["lm_head.weight"], cfg["vocab"], d["H"]).T / a[1]).ravel()


# T around the 8-token attention tile and past a batch of 256; contexts of one and of several key ranges, ragged
@pytest.mark.parametrize("T,P", [(2, 0), (8, 3), (9, 590), (17, 250), (64, 41), (258, 40)])
def test_bonsai_prompt_layer_against_64_bits(ctx, T, P):
    cfg = dict(layers=2, hidden=1024, intermediate=2048, n_heads=8, n_kv_heads=4, head_dim=HD, vocab=512, rope_theta=THETA,
               rms_eps=EPS, max_ctx=P + T + 1)
    W = B.make_weights(cfg, 21)
    rng = np.random.default_rng(T + P)
    for l in range(2):
        W["model.layers.%d.self_attn.q_norm.weight" % l] *= np.float32(3.0)
    pre = [[rng.standard_normal((P, 512)).astype(np.float32) for _ in range(2)] for _ in range(2)]
    ids = rng.integers(0, cfg["vocab"], T).astype(np.int32)
    m = abi.Bonsai(ctx, **cfg)
    try:
        B.load_into(ctx, m, W, cfg["hidden"])
        for l in range(2):
            for ptr, r in zip(m.kv(l), pre[l]):
                if P:
                    ctx.write(ptr, r)
        m.forward(ids, P)
        got = [[ctx.download(ptr, np.float32, (P + T) * 512).reshape(-1, 512)[P:] for ptr in m.kv(l)] for l in range(2)]
        logits = ctx.download(m.logits_ptr(), np.float32, cfg["vocab"]).astype(np.float64)
    finally:
        m.close()
    rows, want = bonsai_f64(cfg, W, pre, got, ids, P)
    check(got, rows, logits, want)
