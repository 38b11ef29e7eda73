"""What a descriptor's launch runs, as the C ABI and GemmDesc.launches report it
(CPU): the descriptor's own kernel when it was made from a configuration, and
for a plan the kernels chosen in its place, whose compiled waits and register
use are the ones the host's tables state."""
import ctypes
import os
import subprocess

import pytest

import mini_triton_nvgpu_v1_amd as tb
from mini_triton_nvgpu_v1_amd import configs

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _plan(M, N, K, block, stages=2, waves=4, **options):
    return tb.plan_from_mlir(configs.Workload(
        "w", M, N, K, 0, configs.NORMAL, block, num_waves=waves, stages=stages,
        exact_tile=False, **options).mlir())


def test_struct_layout(tmp_path):
    fields = [f for f, _ in tb.LaunchInfo._fields_]
    src = tmp_path / "layout.c"
    src.write_text(
        '#include <stdio.h>\n#include <stddef.h>\n#include "tb_gfx950.h"\n'
        'int main(void) {\n  printf("%zu\\n", sizeof(tb_launch_info));\n'
        + "".join(f'  printf("%zu\\n", offsetof(tb_launch_info, {f.lstrip("_")}));\n'
                  for f in fields) + "  return 0;\n}\n")
    exe = tmp_path / "layout"
    subprocess.run(["gcc", "-I", os.path.join(ROOT, "include"), str(src), "-o", str(exe)],
                   check=True)
    out = [int(x) for x in subprocess.run([str(exe)], check=True, capture_output=True,
                                          text=True).stdout.split()]
    assert out == ([ctypes.sizeof(tb.LaunchInfo)]
                   + [getattr(tb.LaunchInfo, f).offset for f in fields])


def test_configured_descriptor_runs_its_own_kernel():
    d = tb.GemmDesc.from_config(_plan(1000, 1496, 712, (256, 256, 64)).config)
    (one,) = d.launches
    assert one.kernel_name == d.kernel_name == d.launched
    assert one.config == d.config and (one.row0, one.col0) == (0, 0)
    info = tb.LaunchInfo()
    for i in (-1, 1):
        assert tb.lib().tb_desc_launch_info(d._h, i, ctypes.byref(info)) != 0


def test_plan_reports_what_runs():
    d = _plan(1000, 1496, 712, (256, 256, 64), activation="silu")
    assert d.kernel_name == "tb_gemm_gfx950_256x256x64_w2x2_s2_out0_16x16x32_epi"
    assert d.launched == "tb_gemm_gfx950_64x128x64_w2x4_s3_out0_epi"
    d = _plan(4104, 4096, 520, (256, 256, 64))
    first, rest = d.launches
    assert first.kernel_name == d.kernel_name and first.config.m == 4096
    assert (rest.row0, rest.col0, rest.config.m, rest.config.n) == (4096, 0, 8, 4096)


PLANS = [
    (1000, 1496, 712, (256, 256, 64), {}),
    (1000, 1496, 712, (256, 256, 64), {"bias": "f16", "activation": "silu"}),
    (4104, 4096, 520, (256, 256, 64), {"c_f32": True}),
    (300, 520, 5000, (128, 128, 64), {"split_k": 4}),
    (300, 520, 5000, (128, 64, 64), {"split_k": 4}),
    (1000, 776, 4168, (128, 128, 64),
     {"split_k": 4, "c_f32": True,
      "module_attrs": {"tb.reduction-mode": '"split_k_parallel"'}}),
    (900, 1032, 1032, (128, 128, 64), {}),
]


@pytest.mark.parametrize("M,N,K,block,options", PLANS)
def test_launched_kernels_hold_their_registers_and_waits(M, N, K, block, options):
    d = _plan(M, N, K, block, **options)
    assert d.launched != d.kernel_name
    area = 0
    for x in d.launches:
        c = x.config
        assert 0 < x.vgprs and x.vgprs + x.agprs <= 512 and x.scratch_bytes == 0
        # a wait for all but the youngest S-1 (then S-2) k-tiles' loads: rounds
        # of 16 bytes per thread of each operand; the 256x256 kernel waits for
        # everything in its loop
        threads = c.num_waves * 64
        loads = sum(-(-chunks // threads) for chunks in (c.block_m * c.block_k // 8,
                                                         c.block_k * c.block_n // 8))
        hand = c.block_m == c.block_n == 256
        assert x.vmcnt_prologue == (c.stages - 1) * loads
        assert x.vmcnt_loop == (0 if hand else (c.stages - 2) * loads)
        area += c.m * c.n
    assert area == M * N
