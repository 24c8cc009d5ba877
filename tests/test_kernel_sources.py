"""Kernels whose waves hand data from lane to lane through LDS of their own, without a workgroup barrier, fence both sides
of the hand-off: nothing else keeps the compiler from moving a lane's reads above another lane's writes."""
import os

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tabinfer_amd", "csrc")


# the writes into the wave's part of LDS, and the first read of them by other lanes
@pytest.mark.parametrize("name,write,read", [
    ("k_gemm.hip", "L.sw[n][j][m] =", "xs4[t] = *reinterpret_cast<const v4f*>(&L.sx"),
    ("k_moe_gemm.hip", "L.sx[t][j][m] =", "xs4[t] = *reinterpret_cast<const v4f*>(&L.sx"),
    ("k_tern_gemm.hip", "L.act[4 * q + j][r] =", "sc[n] = L.scale["),
    ("k_bonsai_batch.hip", "L.k[2 * i + lr][lp] =", "kk = L.k["),
    ("k_tattn.hip", "store_blk();", "process(wave,"),
])
def test_wave_private_lds_is_fenced(name, write, read):
    src = open(os.path.join(CSRC, name)).read()
    assert src.count(write) == 1
    w = src.index(write)
    r = src.index(read, w)
    fence = "ti_wave_lds_fence();"
    assert fence in src[w:r]                        # written, then read
    loop = max(src.rfind("for (int st", 0, w), src.rfind("for (int tile", 0, w), src.rfind("auto step =", 0, w), src.rfind("while (blk", 0, w))
    assert loop >= 0 and fence in src[loop:w]       # read, then written again
