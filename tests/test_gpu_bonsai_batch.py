"""The Bonsai decoder's T-token forward (Model::forward per prompt token, native/crates/n2-core/src/model.rs:349-501,
as one batch) against the same prompt token by token: KV rows, logits, greedy token, device position."""
import numpy as np
import pytest

from tabinfer_amd import abi
import bonsai_ref as B

pytestmark = pytest.mark.gpu

CFG = dict(layers=2, hidden=1024, intermediate=3072, n_heads=8, n_kv_heads=4, head_dim=128, vocab=1000, rope_theta=1e6,
           rms_eps=1e-6, max_ctx=600)
# The first layer's rows: both paths quantize the same embeddings, normalised in f32; a code that
# stood at its rounding boundary differs by one, which is one of K = 1024 terms of rms 35 codes:
# 1 / (32 * 35 * 0.8) = 1.1e-3 of the projection's rms (0.8: the rms of a ternary code), and the
# largest of its values is above 2 rms.
TOL_FIRST = 1e-3
# Behind it each of the 8 quantized inputs of two layers and the head may have been rounded
# otherwise throughout: an rms of 1 / sqrt(12) code against 35 on either side, sqrt(2 * 8) * 0.289 / 35.
TOL = 0.033


@pytest.fixture(scope="module")
def ctx():
    c = abi.Ctx(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def models(ctx):
    W = B.make_weights(CFG, 11)
    ms = [abi.Bonsai(ctx, **CFG) for _ in range(2)]
    for m in ms:
        B.load_into(ctx, m, W, CFG["hidden"])
    yield ms
    for m in ms:
        m.close()


def state(ctx, m, end):
    nkv = CFG["n_kv_heads"] * 128
    rows = [ctx.download(p, np.float32, end * nkv) for l in range(CFG["layers"]) for p in m.kv(l)]
    return ctx.download(m.logits_ptr(), np.float32, CFG["vocab"]), rows


# T: around the 8-token attention tile and the 16-token GEMM tile, past one batch of 256; the
# context from empty to several key tiles and ranges
@pytest.mark.parametrize("T,pos", [(2, 0), (7, 0), (8, 3), (9, 16), (17, 0), (33, 100), (64, 41), (260, 0), (3, 590)])
def test_forward_of_a_prompt_is_its_tokens_in_turn(ctx, models, T, pos):
    one, many = models
    rng = np.random.default_rng(T + pos)
    pre = rng.standard_normal((2 * CFG["layers"], pos, CFG["n_kv_heads"] * 128)).astype(np.float32)
    ids = rng.integers(0, CFG["vocab"], T).astype(np.int32)
    for m in models:
        for i, p in enumerate(q for l in range(CFG["layers"]) for q in m.kv(l)):
            if pos:
                ctx.write(p, pre[i])
    for t in range(T):
        one.forward(ids[t:t + 1], pos + t)
    many.forward(ids, pos)
    (lo, ro), (lm, rm) = state(ctx, one, pos + T), state(ctx, many, pos + T)
    assert B.rel(lm, lo) < TOL
    for i, (a, b) in enumerate(zip(rm, ro)):
        assert np.array_equal(a[:pre[0].size], b[:pre[0].size])
        assert B.rel(a, b) < (TOL_FIRST if i < 2 else TOL)
    assert int(many.read_tokens(pos + T, 1)[0]) == int(np.argmax(lm))
    many.decode()                                   # the device position is pos + T
    one.write_tokens(pos + T, many.read_tokens(pos + T, 1))
    one.set_pos(pos + T)
    one.decode()
    assert B.rel(state(ctx, many, 0)[0], state(ctx, one, 0)[0]) < TOL


def test_captured_forward_replays_like_eager(ctx, models):
    m = models[1]
    ids = np.arange(5, 25, dtype=np.int32)
    m.forward(ids, 0)
    want = state(ctx, m, 20)[0]
    ctx.sync()
    ctx.graph_begin()
    ctx.call("ti_bonsai_forward", m.h, None, 20, 0)
    g = ctx.graph_end()
    try:
        for _ in range(3):
            m.decode()                              # moves the position and the buffers in between
            ctx.graph_launch(g)
            ctx.sync()
            assert np.array_equal(state(ctx, m, 20)[0], want)
    finally:
        ctx.graph_destroy(g)
