"""Performance cases of libtabinfer: the work its users have it do, through the C ABI's Python
binding (tabinfer_amd.abi), from a one-token MLP block to a 256-token prefill chunk.

A case is a dict of plain values; `kind` picks the path:

  decode        one token of a Qwen3 stack at a cached context, a captured step replayed
  forward       T tokens of a Qwen3 stack at once (a prompt chunk, a batch of drafted tokens)
  mlp           a decode token's MLP block: norm + gate/up + SiLU, down
  attn_step     a decode token's attention layer over the int8 KV cache
  lm_head       final norm + int4 lm_head + argmax
  linear        one int4 projection of T tokens
  attn_causal   the attention of a T-token chunk over the int8 KV cache
  moe_decode    the int3 MoE block of one token
  moe_prefill   the int3 MoE block of T tokens
  tern_gemv     ternary projections of one token that share their input (q/k/v, gate/up)
  tern_gemm     one ternary projection of B tokens
  bonsai        T prompt tokens of a ternary Bonsai stack

The stacks hold a few layers of the model (a change of rounding in one layer moves int8 codes in
all that follow, so a deep stack could not be compared); every other case is one layer or block.
Inputs are synthetic: normal weights and activations through the formats' own quantizers, a
KV cache of unit-variance heads. Sizes are those of the models the repository is configured
for (Qwen3-0.6B / 1.7B, Bonsai-1.7B, LFM2.5-8B-A1B), and ragged ones between.
"""
import math

import torch

from tabinfer_amd import abi

DEV = "cuda"
EPS = 1e-6
THETA = 1e6
VOCAB = 151936


def listed():
    return [
        # the smallest call: a Qwen3-0.6B token's MLP block, bound by launches and latency
        dict(name="mlp_0p6b_token", kind="mlp", hidden=1024, inter=3072),
        # a generated Qwen3-1.7B token at a long-chat context, as generate() replays it
        dict(name="decode_1p7b_8k", kind="decode", layers=4, hidden=2048, inter=6144, heads=16, kv_heads=8, pos=8191),
        # one 256-token chunk of a longer prompt, as generate() prefills it
        dict(name="prefill_1p7b_256", kind="forward", layers=2, hidden=2048, inter=6144, heads=16, kv_heads=8, T=256, pos=1792),
        # attention of one token near the full 32k context, at a ragged position
        dict(name="attn_step_32k", kind="attn_step", heads=16, kv_heads=8, hd=128, pos=32101),
        # the vocabulary projection of one token
        dict(name="lm_head_1p7b", kind="lm_head", N=VOCAB, K=2048),
        # the last, ragged chunk of a prompt through one projection
        dict(name="linear_ragged_77", kind="linear", T=77, N=6144, K=2048),
        # the attention of a whole chunk over a 4k context
        dict(name="attn_causal_256_4k", kind="attn_causal", heads=16, kv_heads=8, hd=128, T=256, pos=3840),
        # a generated token's MoE block, and a prompt's
        dict(name="moe_token", kind="moe_decode", hidden=2048, inter=1792, experts=32, topk=4),
        dict(name="moe_prompt_128", kind="moe_prefill", hidden=2048, inter=1792, experts=32, topk=4, T=128),
        # Bonsai-1.7B: gate/up of a generated token; down of a prompt's tokens; a prompt through the decoder
        dict(name="tern_gate_up_token", kind="tern_gemv", K=2048, N0=6144, N1=6144, N2=0),
        dict(name="tern_down_50", kind="tern_gemm", N=2048, K=6144, B=50),
        dict(name="bonsai_prompt_48", kind="bonsai", layers=2, hidden=2048, inter=6144, heads=16, kv_heads=8, T=48, pos=100),
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["mlp", "decode", "forward", "forward", "attn_step", "lm_head", "linear", "linear", "attn_causal",
                       "moe_decode", "moe_prefill", "tern_gemv", "tern_gemm", "bonsai"])
    hidden, inter = rng.choice([(1024, 3072), (2048, 6144)])
    heads = dict(heads=16, kv_heads=8)
    if kind == "mlp":
        return dict(kind=kind, hidden=rng.choice([512, 768, 1024, 1024, 1536, 2048, 2048, 3072]), inter=32 * rng.randint(32, 240))
    if kind == "decode":
        return dict(kind=kind, layers=rng.randint(2, 4), hidden=hidden, inter=inter, pos=_log(rng, 32, 30000), **heads)
    if kind == "forward":
        return dict(kind=kind, layers=2, hidden=hidden, inter=inter, T=_log(rng, 2, 256),
                    pos=rng.choice([0, _log(rng, 1, 4000)]), **heads)
    if kind == "attn_step":
        nh, nkv = rng.choice([(16, 8), (8, 8), (8, 4)])
        return dict(kind=kind, heads=nh, kv_heads=nkv, hd=rng.choice([64, 128, 128]), pos=_log(rng, 32, 32767))
    if kind == "lm_head":
        return dict(kind=kind, N=_log(rng, 2000, VOCAB), K=rng.choice([512, 1024, 2048, 4096]))
    if kind == "linear":
        return dict(kind=kind, T=_log(rng, 2, 256), N=_log(rng, 64, 8192), K=32 * _log(rng, 8, 200))
    if kind == "attn_causal":
        nh, nkv = rng.choice([(16, 8), (8, 8), (16, 4)])
        return dict(kind=kind, heads=nh, kv_heads=nkv, hd=128, T=_log(rng, 2, 256), pos=rng.choice([0, _log(rng, 16, 6000)]))
    if kind == "moe_decode":
        return dict(kind=kind, hidden=rng.choice([2048, 32 * rng.randint(16, 64)]), inter=32 * rng.randint(16, 64),
                    experts=rng.choice([8, 16, 32]), topk=rng.choice([2, 4]))
    if kind == "moe_prefill":
        return dict(kind=kind, hidden=rng.choice([2048, 32 * rng.randint(16, 64)]),
                    inter=rng.choice([1792, 32 * rng.randint(16, 64)]), experts=rng.choice([8, 16, 32]),
                    topk=rng.choice([2, 4]), T=_log(rng, 2, 160))
    if kind == "tern_gemv":
        a, b = rng.randint(500, 9000), rng.randint(500, 2500)
        a, b, c = rng.choice([(a, a, 0), (a, b, b), (a, 0, 0)])
        return dict(kind=kind, K=1024 * rng.randint(1, 6), N0=a, N1=b, N2=c)
    if kind == "tern_gemm":
        return dict(kind=kind, N=_log(rng, 256, 8192), K=rng.choice([2048, 6144, 64 * rng.randint(8, 100)]), B=_log(rng, 2, 128))
    return dict(kind="bonsai", layers=2, hidden=2048, inter=6144, T=_log(rng, 2, 48), pos=rng.choice([0, _log(rng, 1, 900)]), **heads)


# ---- synthetic tensors (the same for prepare() and exact()) --------------------------------
class Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed) * 2654435761 % (1 << 62) + 17)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device=DEV) * std

    def uniform(self, lo, hi, *shape):
        return torch.rand(*shape, generator=self.g, device=DEV) * (hi - lo) + lo

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device=DEV)

    def norm_w(self, n):
        return (1.0 + 0.1 * self.normal(n)).half()

    def int4(self, n, k, std=0.02):
        """Normal weights as int4 groups of 32: packed nibbles (code + 8) and f16 scales."""
        w = self.normal(n, k // 32, 32, std=std)
        s = (w.abs().amax(-1) / 7.0).half()
        q = torch.round(w / s.float().unsqueeze(-1)).clamp_(-8, 7).add_(8).to(torch.uint8).view(n, k)
        return (q[:, 0::2] | (q[:, 1::2] << 4)).contiguous(), s.contiguous()

    def int3(self, rows, k, std=0.02):
        """Normal weights as int3 groups of 32: three bitplanes (code + 4) and f16 scales."""
        w = self.normal(rows, k // 32, 32, std=std)
        s = (w.abs().amax(-1) / 4.0).half()
        q = torch.round(w / s.float().unsqueeze(-1)).clamp_(-4, 3).add_(4).to(torch.uint8)
        bit = torch.arange(8, device=DEV, dtype=torch.uint8)
        planes = [(((q >> b) & 1).view(rows, k // 32, 4, 8) << bit).sum(-1, dtype=torch.uint8) for b in range(3)]
        return torch.stack(planes, 2).contiguous(), s.contiguous()

    def tern(self, n, k):
        """Uniform ternary codes in blocks of 64 (code c at byte c & 15, bits 2 (c >> 4)), f32 scales."""
        c = self.ints(0, 3, n, k // 64, 4, 16).to(torch.uint8)
        b = c[:, :, 0] | (c[:, :, 1] << 2) | (c[:, :, 2] << 4) | (c[:, :, 3] << 6)
        return b.contiguous(), self.uniform(0.01, 0.05, n, k // 64).half().float().contiguous()

    def kv(self, s, nkv, hd):
        """Cached heads: int8 codes [s][nkv][hd] and their per-32 scales."""
        x = self.normal(s, nkv, hd // 32, 32)
        m = x.abs().amax(-1)
        c = torch.floor(0.5 + 127.0 * (x / m.unsqueeze(-1))).to(torch.int8).view(s, nkv, hd)
        return c.contiguous(), m.contiguous()


def _f64_int4(w):
    p, s = w
    q = torch.stack([p & 15, p >> 4], -1).view(p.shape[0], -1, 32)
    return ((q.double() - 8.0) * s.double().unsqueeze(-1)).view(p.shape[0], -1)


def _f64_int3(w):
    p, s = w
    bit = torch.arange(8, device=DEV, dtype=torch.uint8)
    b = ((p.unsqueeze(-1) >> bit) & 1).view(*p.shape[:3], 32).double()
    return ((b[:, :, 0] + 2 * b[:, :, 1] + 4 * b[:, :, 2] - 4.0) * s.double().unsqueeze(-1)).view(p.shape[0], -1)


def _f64_tern(w):
    b, s = w
    c = torch.stack([b & 3, (b >> 2) & 3, (b >> 4) & 3, b >> 6], 2).view(b.shape[0], b.shape[1], 64)
    return ((c.double() - 1.0) * s.double().unsqueeze(-1)).view(b.shape[0], -1)


def _f64_kv(cs):
    c, s = cs
    return (c.double().view(*s.shape, 32) * (s.double() / 127.0).unsqueeze(-1)).view(c.shape)


def _q8(x):
    """The int8 activation of quantQ8 (per 32: absmax / 127, nearest even) as the values it stands for."""
    v = x.float().reshape(-1, 32)
    s = v.abs().amax(-1, keepdim=True) / 127.0
    inv = torch.where(s > 0, 1.0 / s, torch.zeros_like(s))
    return (torch.round(v * inv).clamp(-127, 127).double() * s.double()).view(x.shape)


def _n2(x):
    """quantize_act: per-tensor int8 codes (127 / absmax, nearest, halves away from zero) per row, and the scale."""
    v = x.float()
    s = 127.0 / v.abs().amax(-1, keepdim=True)
    y = v * s
    return (torch.sign(y) * torch.floor(y.abs() + 0.5)).clamp(-127, 127).double(), s.double()


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, pos0, f32_angles=False):
    """Split-half rotary embedding of x [T][heads][hd] at pos0.."""
    T, _, hd = x.shape
    i = torch.arange(hd // 2, device=DEV)
    p = torch.arange(pos0, pos0 + T, device=DEV)
    if f32_angles:
        a = (p.float()[:, None] * torch.pow(torch.tensor(THETA, device=DEV), -(2 * i).float() / hd)[None]).double()
    else:
        a = p.double()[:, None] * torch.pow(torch.tensor(THETA, dtype=torch.float64, device=DEV), -2.0 * i.double() / hd)[None]
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    lo, hi = x[..., : hd // 2], x[..., hd // 2:]
    return torch.cat([lo * c - hi * s, hi * c + lo * s], -1)


def _snorm(x):
    """The KV cache's int8 rows of x [T][heads][hd]: codes, scales."""
    v = x.float().view(*x.shape[:-1], -1, 32)
    m = v.abs().amax(-1).clamp(min=1e-12)
    c = torch.floor(0.5 + 127.0 * (v / m.unsqueeze(-1)).clamp(-1, 1).double()).to(torch.int8)
    return c.view(x.shape), m


def _attend(q, k, v, pos0):
    """q [T][nHq][hd] at positions pos0.. over k, v [S][nKv][hd], causal."""
    T, nq, hd = q.shape
    S, nkv, _ = k.shape
    g = nq // nkv
    mask = torch.arange(S, device=DEV)[None] > (pos0 + torch.arange(T, device=DEV))[:, None]
    out = torch.empty_like(q)
    for h in range(nq):
        s = q[:, h] @ k[:, h // g].t().contiguous() / math.sqrt(hd)
        out[:, h] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ v[:, h // g].contiguous()
    return out


def _silu_mul(g, u):
    return g / (1.0 + torch.exp(-g)) * u


# ---- the library ------------------------------------------------------------------------------
_CTX = []


def _ctx():
    """The program's one context (one stream), made on first use and kept."""
    if not _CTX:
        _CTX.append(abi.Ctx(0))
    return _CTX[0]


class _Mem:
    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (int(ptr), False), "version": 2}


def _view(owner, ptr, shape, typestr):
    """A tensor over device memory of `owner` (a _Stack), which lives as long as the tensor does."""
    return torch.as_tensor(_Mem(owner, ptr, shape, typestr), device=DEV)


def _p(t):
    return t.data_ptr()


def _zeros(*shape, dtype=torch.float32):
    return torch.zeros(*shape, dtype=dtype, device=DEV)


class _Stack:
    """A decoder and its captured step, released with the state that holds it."""

    def __init__(self, model):
        self.m, self.graph = model, None

    def __del__(self):
        ctx = _ctx()
        ctx.sync()
        if self.graph is not None:
            ctx.graph_destroy(self.graph)
        self.m.close()


def _qwen_shapes(c):
    hd = 128
    nq, nkv, H, I = c["heads"] * hd, c["kv_heads"] * hd, c["hidden"], c["inter"]
    return {"self_attn.q_proj": (nq, H), "self_attn.k_proj": (nkv, H), "self_attn.v_proj": (nkv, H),
            "self_attn.o_proj": (H, nq), "mlp.gate_proj": (I, H), "mlp.up_proj": (I, H), "mlp.down_proj": (H, I)}


def _qwen_inputs(c, seed):
    r = Rand(seed)
    T = c.get("T", 1)
    w = {"embed": (r.normal(VOCAB, c["hidden"], std=0.5)).half(), "norm": r.norm_w(c["hidden"]), "lm": r.int4(VOCAB, c["hidden"]),
         "ids": r.ints(0, VOCAB, T).to(torch.int32), "layers": []}
    for _ in range(c["layers"]):
        y = {n: r.int4(*s) for n, s in _qwen_shapes(c).items()}
        y.update({"input_layernorm": r.norm_w(c["hidden"]), "post_attention_layernorm": r.norm_w(c["hidden"]),
                  "self_attn.q_norm": r.norm_w(128), "self_attn.k_norm": r.norm_w(128)})
        y["k"], y["v"] = r.kv(c["pos"], c["kv_heads"], 128), r.kv(c["pos"], c["kv_heads"], 128)
        w["layers"].append(y)
    return w


def _prepare_qwen(c, seed):
    ctx, w = _ctx(), _qwen_inputs(c, seed)
    T, pos, nkv = c.get("T", 1), c["pos"], c["kv_heads"]
    cap = pos + T + 8
    st = _Stack(abi.Qwen3(ctx, layers=c["layers"], hidden=c["hidden"], intermediate=c["inter"], n_heads=c["heads"],
                          n_kv_heads=nkv, head_dim=128, vocab=VOCAB, rope_theta=THETA, rms_eps=EPS, max_ctx=cap,
                          max_tokens=T))
    m = st.m

    def put(name, val):
        d, nd, s, ns = m.tensor(name)
        data, scales = val if isinstance(val, tuple) else (val, None)
        _view(st, d, (nd,), "|u1").copy_(data.contiguous().view(torch.uint8).view(-1))
        if scales is not None:
            _view(st, s, (ns,), "|u1").copy_(scales.contiguous().view(torch.uint8).view(-1))

    put("model.embed_tokens.weight", w["embed"])
    put("model.norm.weight", w["norm"])
    put("lm_head.weight", w["lm"])
    out = {"logits": _view(st, m.logits_ptr(), (VOCAB,), "<f4")}
    slots = m.kv_slots()
    for l, y in enumerate(w["layers"]):
        for n in list(_qwen_shapes(c)) + ["input_layernorm", "post_attention_layernorm", "self_attn.q_norm", "self_attn.k_norm"]:
            put("model.layers.%d.%s.weight" % (l, n), y[n])
        kq, ks, vq, vs = m.kv(l)
        for part, codes, scales, rows in (("k", kq, ks, y["k"]), ("v", vq, vs, y["v"])):
            cv, sv = _view(st, codes, (cap, slots, 128), "|i1"), _view(st, scales, (cap, nkv, 4), "<f4")
            cv[:pos, :nkv].copy_(rows[0])
            sv[:pos].copy_(rows[1])
            # the cache rows this pass writes; past the first layer the codes stand at their rounding
            # boundaries for another rounding of the layers before, so there the scales alone
            if l == 0:
                out["%s%d_codes" % (part, l)] = cv[pos:pos + T, :nkv]
            out["%s%d_scales" % (part, l)] = sv[pos:pos + T]
    ids = w["ids"].cpu().numpy()
    torch.cuda.synchronize()
    state = {"kind": c["kind"], "stack": st, "out": out, "ids": ids, "pos": pos}
    if c["kind"] == "decode":
        m.write_tokens(pos, ids)
        m.set_pos(pos)
        ctx.graph_begin()
        m.decode()
        st.graph = ctx.graph_end()
    return state


def _exact_qwen(c, seed):
    w, T, pos, hd = _qwen_inputs(c, seed), c.get("T", 1), c["pos"], 128
    x = w["embed"][w["ids"].long()].double()
    out = {}
    for l, y in enumerate(w["layers"]):
        a = _q8(_rms(x, y["input_layernorm"]))
        q, k, v = [(a @ _f64_int4(y["self_attn.%s_proj" % n]).t().contiguous()).view(T, -1, hd) for n in "qkv"]
        q, k = _rope(_rms(q, y["self_attn.q_norm"]), pos), _rope(_rms(k, y["self_attn.k_norm"]), pos)
        kc, vc = _snorm(k), _snorm(v)
        for part, rows in (("k", kc), ("v", vc)):
            if l == 0:
                out["%s%d_codes" % (part, l)] = None
            out["%s%d_scales" % (part, l)] = rows[1].double()
        keys, vals = torch.cat([_f64_kv(y["k"]), _f64_kv(kc)]), torch.cat([_f64_kv(y["v"]), _f64_kv(vc)])
        o = _attend(q, keys, vals, pos).reshape(T, -1)
        x = x + _q8(o) @ _f64_int4(y["self_attn.o_proj"]).t().contiguous()
        a = _q8(_rms(x, y["post_attention_layernorm"]))
        g, u = [a @ _f64_int4(y["mlp.%s_proj" % n]).t().contiguous() for n in ("gate", "up")]
        x = x + _q8(_silu_mul(g, u)) @ _f64_int4(y["mlp.down_proj"]).t().contiguous()
    out["logits"] = (_f64_int4(w["lm"]) @ _rms(x[-1], w["norm"]).unsqueeze(-1)).squeeze(-1)
    return out


BONSAI = {"self_attn.q_proj": ("nq", "H"), "self_attn.k_proj": ("nkv", "H"), "self_attn.v_proj": ("nkv", "H"),
          "self_attn.o_proj": ("H", "nq"), "mlp.gate_proj": ("I", "H"), "mlp.up_proj": ("I", "H"), "mlp.down_proj": ("H", "I")}


def _bonsai_inputs(c, seed):
    r, H, hd = Rand(seed), c["hidden"], 128
    d = {"nq": c["heads"] * hd, "nkv": c["kv_heads"] * hd, "H": H, "I": c["inter"]}
    w = {"embed": r.normal(VOCAB, H, std=0.5).half(), "norm": r.norm_w(H).float(), "lm": r.tern(VOCAB, H),
         "ids": r.ints(0, VOCAB, c["T"]).to(torch.int32), "layers": []}
    for _ in range(c["layers"]):
        y = {n: r.tern(d[a], d[b]) for n, (a, b) in BONSAI.items()}
        y.update({"input_layernorm": r.norm_w(H).float(), "post_attention_layernorm": r.norm_w(H).float(),
                  "self_attn.q_norm": r.norm_w(hd).float(), "self_attn.k_norm": r.norm_w(hd).float(),
                  "k": r.normal(c["pos"], d["nkv"]), "v": r.normal(c["pos"], d["nkv"])})
        w["layers"].append(y)
    return w


def _prepare_bonsai(c, seed):
    ctx, w, T, pos = _ctx(), _bonsai_inputs(c, seed), c["T"], c["pos"]
    nkv, cap = c["kv_heads"] * 128, 1024
    st = _Stack(abi.Bonsai(ctx, layers=c["layers"], hidden=c["hidden"], intermediate=c["inter"], n_heads=c["heads"],
                           n_kv_heads=c["kv_heads"], head_dim=128, vocab=VOCAB, rope_theta=THETA, rms_eps=EPS, max_ctx=cap))
    m = st.m

    def put(name, val):
        d, nd, s, ns = m.tensor(name)
        data, scales = val if isinstance(val, tuple) else (val, None)
        _view(st, d, (nd,), "|u1").copy_(data.view(torch.uint8).view(-1))
        if scales is not None:
            _view(st, s, (ns,), "|u1").copy_(scales.view(torch.uint8).view(-1))

    put("model.embed_tokens.weight", w["embed"])
    put("model.norm.weight", w["norm"])
    put("lm_head.weight", w["lm"])
    out = {"logits": _view(st, m.logits_ptr(), (VOCAB,), "<f4")}
    for l, y in enumerate(w["layers"]):
        for n in list(BONSAI) + ["input_layernorm", "post_attention_layernorm", "self_attn.q_norm", "self_attn.k_norm"]:
            put("model.layers.%d.%s.weight" % (l, n), y[n])
        for part, ptr in zip("kv", m.kv(l)):
            rows = _view(st, ptr, (cap, nkv), "<f4")
            rows[:pos].copy_(y[part])
            out["%s%d" % (part, l)] = rows[pos:pos + T]
    ids = w["ids"].cpu().numpy()
    torch.cuda.synchronize()
    return {"kind": c["kind"], "stack": st, "out": out, "ids": ids, "pos": pos}


def _exact_bonsai(c, seed):
    w, T, pos, hd = _bonsai_inputs(c, seed), c["T"], c["pos"], 128
    x = w["embed"][w["ids"].long()].double()
    out = {}

    def lin(a, weight):
        codes, s = a
        return codes @ _f64_tern(weight).t().contiguous() / s

    for l, y in enumerate(w["layers"]):
        a = _n2(_rms(x, y["input_layernorm"]))
        q, k, v = [lin(a, y["self_attn.%s_proj" % n]).view(T, -1, hd) for n in "qkv"]
        q = _rope(_rms(q, y["self_attn.q_norm"]), pos, True)
        k = _rope(_rms(k, y["self_attn.k_norm"]), pos, True)
        out["k%d" % l], out["v%d" % l] = k.reshape(T, -1), v.reshape(T, -1)
        keys = torch.cat([y["k"].double(), out["k%d" % l]]).view(pos + T, -1, hd)
        vals = torch.cat([y["v"].double(), out["v%d" % l]]).view(pos + T, -1, hd)
        x = x + lin(_n2(_attend(q, keys, vals, pos).reshape(T, -1)), y["self_attn.o_proj"])
        a = _n2(_rms(x, y["post_attention_layernorm"]))
        x = x + lin(_n2(_silu_mul(lin(a, y["mlp.gate_proj"]), lin(a, y["mlp.up_proj"]))), y["mlp.down_proj"])
    out["logits"] = lin(_n2(_rms(x[-1:], w["norm"])), w["lm"]).view(-1)
    return out


def _inputs(c, seed):
    """The tensors of the single-layer cases."""
    r, kind = Rand(seed), c["kind"]
    if kind == "mlp":
        H, I = c["hidden"], c["inter"]
        return dict(x=r.normal(H), norm=r.norm_w(H), gate=r.int4(I, H), up=r.int4(I, H), down=r.int4(H, I))
    if kind == "attn_step":
        nh, nkv, hd, pos = c["heads"], c["kv_heads"], c["hd"], c["pos"]
        return dict(q=r.normal(nh, hd), k=r.normal(nkv, hd), v=r.normal(nkv, hd), qn=r.norm_w(hd), kn=r.norm_w(hd),
                    K=r.kv(pos + 1, nkv, hd), V=r.kv(pos + 1, nkv, hd))
    if kind == "lm_head":
        return dict(x=r.normal(c["K"]), norm=r.norm_w(c["K"]), w=r.int4(c["N"], c["K"]))
    if kind == "linear":
        return dict(x=r.normal(c["T"], c["K"]), w=r.int4(c["N"], c["K"]))
    if kind == "attn_causal":
        S = c["pos"] + c["T"]
        return dict(q=r.normal(c["T"], c["heads"], c["hd"]), K=r.kv(S, c["kv_heads"], c["hd"]), V=r.kv(S, c["kv_heads"], c["hd"]))
    if kind in ("moe_decode", "moe_prefill"):
        H, I, nE, T = c["hidden"], c["inter"], c["experts"], c.get("T", 1)
        return dict(x=r.normal(T, H), normed=r.normal(T, H), logits=r.normal(T, nE), bias=r.normal(nE, std=0.1),
                    w1=r.int3(nE * I, H), w3=r.int3(nE * I, H), w2=r.int3(nE * H, I))
    if kind == "tern_gemv":
        a = r.ints(-127, 128, 1, c["K"])
        return dict(a=a, w=[r.tern(n, c["K"]) for n in (c["N0"], c["N1"], c["N2"]) if n])
    return dict(a=r.ints(-127, 128, c["B"], c["K"]), w=r.tern(c["N"], c["K"]))


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("decode", "forward"):
        return _prepare_qwen(c, seed)
    if kind == "bonsai":
        return _prepare_bonsai(c, seed)
    s = _inputs(c, seed)
    s.update(kind=kind, case=c)
    if kind == "mlp":
        s.update(swq=_zeros(c["inter"], dtype=torch.int8), sws=_zeros(c["inter"] // 32), y=_zeros(c["hidden"]))
    elif kind == "attn_step":
        s.update(out=_zeros(c["heads"], c["hd"]), oq=_zeros(c["heads"], c["hd"], dtype=torch.int8), os=_zeros(c["heads"], c["hd"] // 32))
    elif kind == "lm_head":
        s.update(logits=_zeros(c["N"]), hist=_zeros(2, dtype=torch.int32))
    elif kind == "linear":
        s.update(y=_zeros(c["T"], c["N"]))
    elif kind == "attn_causal":
        s.update(out=_zeros(c["T"], c["heads"], c["hd"]))
    elif kind in ("moe_decode", "moe_prefill"):
        P = c.get("T", 1) * c["topk"]
        s.update(res=s["x"].clone(), idx=_zeros(P, dtype=torch.int32), wt=_zeros(P), gate=_zeros(P, c["inter"]),
                 up=_zeros(P, c["inter"]), act=_zeros(P, c["inter"]), out=_zeros(P, c["hidden"]))
    else:
        a = s["a"]
        s["xsum"] = a.view(a.shape[0], -1, 64).sum(-1).to(torch.int32).contiguous()
        s["act"] = a.to(torch.int8).contiguous()
        if kind == "tern_gemv":
            s["y"] = [_zeros(w[1].shape[0]) for w in s["w"]]
            n = len(s["w"])
            ptrs = lambda v: (abi.C.c_void_p * n)(*[_p(t) for t in v])  # noqa: E731
            s["args"] = (ptrs([w[0] for w in s["w"]]), ptrs([w[1] for w in s["w"]]), ptrs(s["y"]),
                         (abi.C.c_int * n)(*[w[1].shape[0] for w in s["w"]]))
        else:
            s["y"] = _zeros(c["B"], c["N"])
    torch.cuda.synchronize()
    return s


def run(s):
    ctx, kind = _ctx(), s["kind"]
    if kind == "decode":
        s["stack"].m.set_pos(s["pos"])
        ctx.graph_launch(s["stack"].graph)
        return s["out"]
    if kind in ("forward", "bonsai"):
        s["stack"].m.forward(s["ids"], s["pos"])
        return s["out"]
    c = s["case"]
    if kind == "mlp":
        H, I = c["hidden"], c["inter"]
        ctx.call("ti_rmsnorm_gateup_silu_q4", _p(s["x"]), _p(s["norm"]), EPS, _p(s["gate"][0]), _p(s["gate"][1]), _p(s["up"][0]),
                 _p(s["up"][1]), None, I, H, _p(s["swq"]), _p(s["sws"]))
        ctx.call("ti_gemv_q4_q8", _p(s["swq"]), _p(s["sws"]), _p(s["down"][0]), _p(s["down"][1]), _p(s["y"]), H, I, 0)
        return {"swi_scales": s["sws"], "y": s["y"]}
    if kind == "attn_step":
        (kc, ks), (vc, vs) = s["K"], s["V"]
        ctx.call("ti_attn_step_q8", _p(s["q"]), _p(s["k"]), _p(s["v"]), _p(s["qn"]), _p(s["kn"]), _p(kc), _p(ks), _p(vc), _p(vs),
                 _p(s["out"]), c["heads"], c["kv_heads"], c["hd"], c["pos"], c["pos"] + 1, THETA, EPS, 0, _p(s["oq"]), _p(s["os"]))
        return {"out": s["out"], "out_scales": s["os"], "k_codes": kc[-1], "k_scales": ks[-1], "v_codes": vc[-1], "v_scales": vs[-1]}
    if kind == "lm_head":
        ctx.call("ti_rmsnorm_lm_head_argmax", _p(s["x"]), _p(s["norm"]), EPS, _p(s["w"][0]), _p(s["w"][1]), _p(s["logits"]),
                 c["N"], c["K"], _p(s["hist"]), 1)
        return {"logits": s["logits"], "token": s["hist"][1:]}
    if kind == "linear":
        ctx.call("ti_linear_q4", _p(s["x"]), _p(s["w"][0]), _p(s["w"][1]), _p(s["y"]), c["T"], c["N"], c["K"], 0)
        return s["y"]
    if kind == "attn_causal":
        ctx.call("ti_attn_causal_q8", _p(s["q"]), _p(s["K"][0]), _p(s["K"][1]), _p(s["V"][0]), _p(s["V"][1]), _p(s["out"]),
                 c["T"], c["pos"], c["heads"], c["kv_heads"], c["hd"])
        return s["out"]
    if kind in ("moe_decode", "moe_prefill"):
        H, I, nE, k = c["hidden"], c["inter"], c["experts"], c["topk"]
        # the block adds to the residual stream, which the layer before has just written
        ctx.call("ti_buf_copy", _p(s["res"]), 0, _p(s["x"]), 0, s["x"].numel() * 4)
        w = [_p(t) for n in ("w1", "w3", "w2") for t in s[n]]
        if kind == "moe_decode":
            ctx.call("ti_moe_decode_q3", _p(s["res"]), _p(s["normed"]), _p(s["logits"]), _p(s["bias"]), *w, _p(s["idx"]),
                     _p(s["wt"]), _p(s["act"]), H, I, nE, k)
        else:
            ctx.call("ti_moe_prefill_q3", _p(s["res"]), _p(s["normed"]), _p(s["logits"]), _p(s["bias"]), *w, _p(s["idx"]),
                     _p(s["wt"]), _p(s["gate"]), _p(s["up"]), _p(s["act"]), _p(s["out"]), c["T"], H, I, nE, k)
        return {"x": s["res"], "experts": s["idx"], "weights": s["wt"]}
    if kind == "tern_gemv":
        codes, scales, outs, Ns = s["args"]
        ctx.call("ti_tern_gemv_multi", _p(s["act"]), _p(s["xsum"]), c["K"], len(s["w"]), codes, scales, outs, Ns)
        return s["y"]
    ctx.call("ti_tern_gemm", _p(s["y"]), c["N"], _p(s["w"][0]), _p(s["w"][1]), _p(s["act"]), _p(s["xsum"]), c["N"], c["K"], c["B"])
    return s["y"]


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("decode", "forward"):
        return _exact_qwen(c, seed)
    if kind == "bonsai":
        return _exact_bonsai(c, seed)
    s = _inputs(c, seed)
    if kind == "mlp":
        a = _q8(_rms(s["x"].double(), s["norm"]))
        swi = _silu_mul(_f64_int4(s["gate"]) @ a, _f64_int4(s["up"]) @ a)
        return {"swi_scales": swi.view(-1, 32).abs().amax(-1) / 127.0, "y": _f64_int4(s["down"]) @ _q8(swi)}
    if kind == "attn_step":
        q = _rope(_rms(s["q"].double(), s["qn"])[None], c["pos"])
        kc, vc = _snorm(_rope(_rms(s["k"].double(), s["kn"])[None], c["pos"])), _snorm(s["v"][None])
        keys, vals = [torch.cat([_f64_kv(old)[:-1], _f64_kv(new)]) for old, new in ((s["K"], kc), (s["V"], vc))]
        out = _attend(q, keys, vals, c["pos"])[0]
        return {"out": out, "out_scales": out.view(c["heads"], -1, 32).abs().amax(-1) / 127.0, "k_codes": None,
                "k_scales": kc[1][0].double(), "v_codes": None, "v_scales": vc[1][0].double()}
    if kind == "lm_head":
        return {"logits": (_f64_int4(s["w"]) @ _rms(s["x"].double(), s["norm"])), "token": None}
    if kind == "linear":
        return _q8(s["x"]) @ _f64_int4(s["w"]).t().contiguous()
    if kind == "attn_causal":
        return _attend(s["q"].double(), _f64_kv(s["K"]), _f64_kv(s["V"]), c["pos"])
    if kind in ("moe_decode", "moe_prefill"):
        I, H, k = c["inter"], c["hidden"], c["topk"]
        g = torch.sigmoid(s["logits"].double())
        e = torch.topk(g + s["bias"].double(), k, dim=-1).indices
        wt = torch.gather(g, 1, e)
        wt = wt / (wt.sum(-1, keepdim=True) + 1e-6)
        quant = _q8 if kind == "moe_prefill" else (lambda v: v)
        a, x = quant(s["normed"].double()), s["x"].double().clone()
        rows = lambda w, i, n: _f64_int3((w[0][i * n:(i + 1) * n], w[1][i * n:(i + 1) * n]))  # noqa: E731
        for i in range(c["experts"]):
            t, slot = torch.nonzero(e == i, as_tuple=True)
            if not len(t):
                continue
            act = _silu_mul(a[t] @ rows(s["w1"], i, I).t().contiguous(), a[t] @ rows(s["w3"], i, I).t().contiguous())
            x.index_add_(0, t, wt[t, slot, None] * (quant(act) @ rows(s["w2"], i, H).t().contiguous()))
        return {"x": x, "experts": None, "weights": wt.view(-1)}
    a = s["a"].double()
    if kind == "tern_gemv":
        return [_f64_tern(w) @ a[0] for w in s["w"]]
    return a @ _f64_tern(s["w"]).t().contiguous()


def work(case):
    c, kind, T = case, case["kind"], case.get("T", 1)
    int4, int3 = 0.5625, 0.4375
    if kind == "mlp":
        n = 3 * c["hidden"] * c["inter"]
        return {"bytes": n * int4 + 8 * c["hidden"], "flops": 2 * n}
    if kind in ("decode", "forward"):
        lin = sum(a * b for a, b in _qwen_shapes(c).values())
        S, nq, nkv = c["pos"] + T, c["heads"] * 128, c["kv_heads"] * 128
        keys = T * c["pos"] + T * (T + 1) // 2
        return {"bytes": c["layers"] * (lin * int4 + S * nkv * 2.25) + VOCAB * (c["hidden"] * int4 + 4) + T * c["hidden"] * 2,
                "flops": c["layers"] * (2 * T * lin + 4 * keys * nq) + 2 * VOCAB * c["hidden"]}
    if kind == "bonsai":
        d = {"nq": c["heads"] * 128, "nkv": c["kv_heads"] * 128, "H": c["hidden"], "I": c["inter"]}
        lin = sum(d[a] * d[b] for a, b in BONSAI.values())
        keys = T * c["pos"] + T * (T + 1) // 2
        return {"bytes": c["layers"] * (lin * 0.3125 + (c["pos"] + T) * d["nkv"] * 8) + VOCAB * (d["H"] * 0.3125 + 4),
                "flops": c["layers"] * (2 * T * lin + 4 * keys * d["nq"]) + 2 * VOCAB * d["H"]}
    if kind == "attn_step":
        kv = (c["pos"] + 1) * c["kv_heads"] * c["hd"]
        return {"bytes": kv * 2.25, "flops": 4 * (c["pos"] + 1) * c["heads"] * c["hd"]}
    if kind == "lm_head":
        return {"bytes": c["N"] * (c["K"] * int4 + 4) + 6 * c["K"], "flops": 2 * c["N"] * c["K"]}
    if kind == "linear":
        return {"bytes": c["N"] * c["K"] * int4 + 4 * T * (c["K"] + c["N"]), "flops": 2 * T * c["N"] * c["K"]}
    if kind == "attn_causal":
        keys = T * c["pos"] + T * (T + 1) // 2
        return {"bytes": (c["pos"] + T) * c["kv_heads"] * c["hd"] * 2.25 + 8 * T * c["heads"] * c["hd"],
                "flops": 4 * keys * c["heads"] * c["hd"]}
    if kind in ("moe_decode", "moe_prefill"):
        pairs, nE = T * c["topk"], c["experts"]
        routed = nE * (1.0 - (1.0 - c["topk"] / nE) ** T)   # experts that at least one token goes to
        return {"bytes": routed * 3 * c["hidden"] * c["inter"] * int3 + 12 * T * c["hidden"], "flops": 6 * pairs * c["hidden"] * c["inter"]}
    if kind == "tern_gemv":
        n = (c["N0"] + c["N1"] + c["N2"]) * c["K"]
        return {"bytes": n * 0.3125 + c["K"] + 4 * n // c["K"], "flops": 2 * n}
    n = c["N"] * c["K"]
    return {"bytes": n * 0.3125 + c["B"] * (c["K"] + 4 * c["N"]), "flops": 2 * c["B"] * n}


def tolerance(case):
    kind = case["kind"]
    # a stack's int8 codes move at their rounding boundaries with the f32 rounding before them, and
    # one moved code moves others in every layer after it (logits against 64 bits: 4e-3 to 1.2e-2 off
    # after 4 decoded layers, 1e-2 after 2 layers of 256 tokens, 1.8e-2 after 2 ternary layers)
    if kind in ("decode", "forward", "bonsai"):
        return {"rel": 0.03, "max": 0.5, "differ": 0.005}
    # the quantized SwiGLU: a moved code is 1 / 127 of its group's largest (9e-6 off over 128 tokens)
    if kind in ("mlp", "moe_prefill"):
        return {"rel": 1e-4, "max": 0.02}
    # f32 sums of exact products: 1e-7 to 3e-7 off
    return {"rel": 2e-6, "max": 1e-4}
