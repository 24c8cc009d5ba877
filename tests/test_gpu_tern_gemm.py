"""The matrix-core ternary GEMM (gemm_tern_b4, cpu/kernel/src/lib.rs:331-367) at the edges of its
tiles: each f32 sum of s * (dot - xsum) against 64 bits, and no further from it than the scalar
gemv_tern (native/crates/n2-kernels/src/tern.rs:79-119), whose two sums cancel."""
import numpy as np
import pytest

from tabinfer_amd import abi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = abi.Ctx(0)
    yield c
    c.close()


def _tern(rng, n, k):
    codes = rng.integers(0, 3, (n * k // 64, 4, 16), dtype=np.uint8)
    packed = codes[:, 0] | (codes[:, 1] << 2) | (codes[:, 2] << 4) | (codes[:, 3] << 6)
    return packed.ravel(), rng.uniform(-0.05, 0.05, n * k // 64).astype(np.float32)


# K: one block, a remainder of the four-block step, fewer steps than waves, whole rounds of them;
# N and B: one below, at and above a 16-wide tile
@pytest.mark.parametrize("n,k,b", [(1, 64, 5), (15, 128, 15), (16, 320, 16), (17, 576, 17), (33, 832, 33), (100, 2048, 50),
                                   (40, 6144, 5), (5000, 1088, 31), (70000, 64, 7), (9000, 2048, 128)])
def test_tern_gemm_against_64_bits(ctx, orc, n, k, b):
    rng = np.random.default_rng(n + k + b)
    codes, sc = _tern(rng, n, k)
    act = rng.integers(-127, 128, (b, k)).astype(np.int8)
    xsum = act.reshape(b, -1, 64).astype(np.int32).sum(-1).astype(np.int32)
    xsum[0] += 3                                    # the caller's sums are used as they are given
    stride = n + 5
    dc, ds, da, dx = ctx.upload(codes), ctx.upload(sc), ctx.upload(act), ctx.upload(xsum)
    dout = ctx.upload(np.full(b * stride, 7.0, np.float32))
    ctx.call("ti_tern_gemm", dout, stride, dc, ds, da, dx, n, k, b)
    out = ctx.download(dout, np.float32, b * stride).reshape(b, stride)
    for x in (dc, ds, da, dx, dout):
        x.free()
    assert np.all(out[:, n:] == 7.0)
    nb = k // 64
    for t in sorted({0, 1, b // 2, b - 1}):
        dots = orc.tern_block_dots(codes, act[t], n, k).reshape(n, nb).astype(np.float64) - xsum[t]
        terms = dots * sc.reshape(n, nb).astype(np.float64)
        ref = terms.sum(1)
        # nb products and sums, each rounded once to 2^-24 of a partial sum no larger than sum |terms|
        assert np.all(np.abs(out[t, :n] - ref) <= (nb + 3) * 2.0 ** -24 * np.abs(terms).sum(1)), t
        scalar = orc.tern_gemv_scalar(codes, sc, act[t], xsum[t], n, k)
        if n >= 100 and nb > 1:
            assert np.linalg.norm(out[t, :n] - ref) <= np.linalg.norm(scalar - ref)
