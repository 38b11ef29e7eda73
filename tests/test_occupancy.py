"""Registers of the small-wave-tile loop: the copy of the loop body for the
last k-tiles is compiled only where it costs no workgroup per CU that LDS has
room for. The compiler's report of the tiles around that rule, as waves per
SIMD (512 registers per lane and SIMD, allocated in eights; accumulation
registers start at a multiple of four)."""
import pytest

import mini_triton_nvgpu_v1_amd as tb

# instance, waves per SIMD at least
TILES = [
    ("64x64x32_w2x2_s2_out0_epi", 5),
    ("64x128x32_w1x4_s2_out0", 5),
    ("64x128x32_w1x4_s2_out0_epi", 3),
    ("64x128x64_w1x4_s2_out0_epi", 3),
    ("128x64x64_w2x2_s2_out1_epi", 3),
    ("128x128x32_w4x2_s2_out0", 6),
    ("192x64x32_w2x2_s2_out0", 4),
    ("64x256x32_w1x8_s2_out0", 6),
    ("64x256x64_w1x8_s2_out0_epi", 4),
]


@pytest.fixture(scope="module")
def resources():
    return tb.kernel_resources()


@pytest.mark.parametrize("name,waves", TILES, ids=[t[0] for t in TILES])
def test_waves_per_simd(name, waves, resources):
    vgprs, agprs, scratch = resources["tb_gemm_gfx950_" + name]
    regs = -(-vgprs // 4) * 4 + agprs if agprs else vgprs
    assert scratch == 0
    assert 512 // (-(-regs // 8) * 8) >= waves, (vgprs, agprs)
