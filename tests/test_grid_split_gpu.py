"""The launches of a plan whose grid leaves CUs idle, or a last round nearly
empty, run on other tiles or as two rectangles of C. Each result is compared
bit for bit with the planned kernel itself (a descriptor made from the plan's
configuration runs exactly that): a whole problem on a finer tile, on a
coarser one, rows and columns cut off as a second rectangle, ragged in M, N
and K, with a bias row, an f32 C and persistent order; padding past the
result is not written. f32 C += A*B has the planned kernel's bits too unless
that one adds the prior C inside its loop; then its error is no larger."""
import pytest
import torch

import mini_triton_nvgpu_v1_amd as tb
from mini_triton_nvgpu_v1_amd import configs

pytestmark = pytest.mark.gpu

ATOMIC = {"tb.reduction-mode": '"split_k_parallel"'}
BIG, MID, SMALL = (256, 256, 64), (128, 128, 64), (64, 64, 64)
T256, T256x128, T128 = ("256x256x64_w2x2_s2_out{}_16x16x32", "256x128x64_w4x2_s3_out{}_16x16x32",
                        "128x128x64_w2x2_s3_out{}_16x16x32")
T64x128, T64 = "64x128x64_w2x4_s3_out{}", "64x64x64_w2x2_s3_out{}"
SPLIT = "128x128x64_w2x2_s3_out{}_16x16x32_split"
# (M, N, K, block, stages, options, the kernels that run with their first row
# and column)
CASES = [
    # one element row, K below a k-tile
    (1, 8, 8, MID, 3, {}, [(T64, 0, 0)]),
    (129, 136, 72, MID, 2, {"bias": "f16", "activation": "silu"}, [(T64 + "_epi", 0, 0)]),
    (1000, 1496, 712, BIG, 2, {"bias": "f32", "clamp_min": -0.5, "clamp_max": 0.5},
     [(T64x128 + "_epi", 0, 0)]),
    (900, 1032, 1032, MID, 2, {}, [(T64, 0, 0)]),  # 2-stage plan with a long K
    (2048, 2056, 200, SMALL, 2, {}, [(T256x128, 0, 0)]),  # a coarser tile
    (4104, 4096, 520, BIG, 2, {"bias": "f16"},    # 8 rows past a whole round
     [(T256 + "_epi", 0, 0), (T64 + "_epi", 4096, 0)]),
    (512, 40000, 264, BIG, 2, {"bias": "f32"},    # columns cut off
     [(T256 + "_epi", 0, 0), (T128 + "_epi", 0, 32768)]),
    (4200, 4200, 328, BIG, 2, {"persistent": True, "num_ctas": 256},
     [(T256, 0, 0), (T64x128, 3840, 0)]),
    (4200, 4200, 328, BIG, 2, {"c_f32": True}, [(T256, 0, 0), (T64, 3840, 0)]),
    (4104, 4096, 2056, BIG, 2, {"c_f32": True}, [(T256, 0, 0), (T64, 4096, 0)]),
    (700, 1504, 2048, BIG, 2, {"c_f32": True}, [(T64x128, 0, 0)]),  # planned: C in the loop
    (3072, 3072, 1280, MID, 3, {"c_f32": True}, [(T128, 0, 0)]),  # not to 256x256
    (2560, 2560, 1280, MID, 3, {"c_f32": True}, [(T256x128, 0, 0)]),
    (2048, 2048, 2048, SMALL, 3, {"c_f32": True}, [(T128, 0, 0)]),
    # split-K: 3 stages for 2, and 128x128 tiles on the 16x16x32 loop (splits of
    # unequal length, a partial last k-tile, fewer rows than a wave tile)
    (300, 520, 5000, (128, 64, 64), 2, {"split_k": 4, "bias": "f16"},
     [("128x64x64_w4x1_s3_out1", 0, 0)]),
    (300, 520, 5000, MID, 2, {"split_k": 4, "bias": "f16", "activation": "relu"},
     [(SPLIT, 0, 0)]),
    (129, 136, 9224, MID, 3, {"split_k": 16}, [(SPLIT, 0, 0)]),
    (7, 1032, 4096, MID, 2, {"split_k": 7, "c_f32": True}, [(SPLIT, 0, 0)]),
    (1000, 776, 4168, MID, 2, {"split_k": 4, "c_f32": True, "module_attrs": ATOMIC},
     [(SPLIT, 0, 0)]),
    (129, 8, 9000, MID, 4, {"split_k": 3, "c_f32": True, "module_attrs": ATOMIC},
     [(SPLIT, 0, 0)]),
]


@pytest.mark.parametrize("M,N,K,block,stages,options,runs", CASES,
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else None)
def test_matches_planned_kernel(M, N, K, block, stages, options, runs, device):
    print(f"grid split {M}x{N}x{K} {block} {options}", flush=True)
    w = configs.Workload("w", M, N, K, 0, configs.NORMAL, block, num_waves=4, stages=stages,
                         exact_tile=False, **options)
    plan = tb.plan_from_mlir(w.mlir())
    exact = tb.GemmDesc.from_config(plan.config)
    assert exact.launched == exact.kernel_name == plan.kernel_name
    out = int(plan.kernel_name.split("_out")[1][0])
    assert ([(x.kernel_name, x.row0, x.col0) for x in plan.launches]
            == [("tb_gemm_gfx950_" + name.format(out), r, c) for name, r, c in runs])
    g = torch.Generator(device=device).manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g, device=device).half()
    b = (torch.randn(K, N, generator=g, device=device) / K ** 0.5).half()
    bias = None
    if w.bias:
        bias = torch.randn(N, generator=g, device=device,
                           dtype=torch.float16 if w.bias == "f16" else torch.float32)
    got = []
    for desc in (plan, exact):
        # C in the middle of a larger buffer whose ends must stay as they are
        buf = torch.full((M * N + 512,), 3.0, device=device,
                         dtype=torch.float32 if w.c_f32 else torch.float16)
        c = buf[256:256 + M * N].view(M, N)
        ws = torch.empty(max(desc.workspace_bytes, 16), dtype=torch.uint8, device=device)
        desc.launch(a, b, c, ws, bias=bias)
        assert (buf[:256] == 3).all() and (buf[256 + M * N:] == 3).all()
        got.append(c)
    if w.split_k > 1 and w.c_f32 and not w.module_attrs:
        assert torch.equal(got[0], got[1])  # fixed reduction order, C added first
    if w.c_f32 and w.split_k == 1:
        in_loop = block == BIG and K % 64 == 0 and K >= 18 * 64
        if not in_loop:  # the prior C is added last on both
            assert torch.equal(got[0], got[1])
        ref = a.double() @ b.double() + 3
        err = [(c - ref).norm() for c in got]
        assert err[0] <= err[1], err
    elif w.c_f32:
        # atomic splits are added in any order: one rounding of each running
        # sum apart
        mag = a.float().abs() @ b.float().abs() + 3
        assert ((got[0] - got[1]).abs() <= (K + 2) * 2.0 ** -23 * mag).all()
        ref = a.double() @ b.double() + 3
        assert ((got[0] - ref).abs() <= (K + 2) * 2.0 ** -24 * mag).all()
    else:
        assert torch.equal(got[0], got[1])


def test_two_rectangles_in_a_graph(device):
    """A captured launch of two rectangles, replayed with eager work between
    the replays, gives the eager result each time."""
    M, N, K = 4104, 4096, 136
    print(f"grid split graph {M}x{N}x{K}", flush=True)
    w = configs.Workload("w", M, N, K, 0, configs.NORMAL, BIG, num_waves=4, exact_tile=False)
    desc = tb.plan_from_mlir(w.mlir())
    assert len(desc.launches) == 2
    a = torch.randn(M, K, device=device).half()
    b = (torch.randn(K, N, device=device) / K ** 0.5).half()
    c = torch.empty(M, N, device=device, dtype=torch.float16)
    desc.launch(a, b, c)
    eager = c.clone()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        desc.launch(a, b, c, stream=stream)
    for _ in range(3):
        c.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, eager)
