"""Registers of the small-wave-tile loop: the copy of the loop body for the
last k-tiles is compiled only where it costs no workgroup per CU that LDS has
room for. The compiler's report of the tiles around that rule, as waves per
SIMD (512 registers per lane and SIMD, allocated in eights; accumulation
registers start at a multiple of four)."""
import importlib.util
import os

import pytest

import mini_triton_nvgpu_v1_amd as tb

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

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


def test_register_table_reads_every_gemm_kernel():
    """Each GEMM kernel family's mangled name is one the table's parser knows,
    the split-K builds that only launches of a plan bind among them."""
    path = os.path.join(ROOT, "mini_triton_nvgpu_v1_amd", "csrc", "tools", "resource_table.py")
    spec = importlib.util.spec_from_file_location("resource_table", path)
    table = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(table)
    for family, args, mangled in [
            ("gemm_mfma16g_split", (128, 128, 64, 2, 2, 3, 1),
             "Li128ELi128ELi64ELi2ELi2ELi3ELi1E"),
            ("gemm_mfma16g", (128, 128, 64, 2, 2, 3, 0, 1),
             "Li128ELi128ELi64ELi2ELi2ELi3ELi0ELb1E"),
            ("gemm_kernel", (64, 64, 32, 2, 2, 0, 2, -1, 0),
             "Li64ELi64ELi32ELi2ELi2ELi0ELi2ELin1ELb0E")]:
        name = f"_ZN3tbk{len(family)}{family}I{mangled}EEvNS_10GemmParamsE"
        assert table.parse_name(name) == (family, args)
