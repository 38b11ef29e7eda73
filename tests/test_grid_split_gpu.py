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
# (M, N, K, block, stages, options)
CASES = [
    (1, 8, 8, MID, 3, {}),                        # one element row, K below a k-tile
    (129, 136, 72, MID, 2, {"bias": "f16", "activation": "silu"}),
    (1000, 1496, 712, BIG, 2, {"bias": "f32", "clamp_min": -0.5, "clamp_max": 0.5}),
    (900, 1032, 1032, MID, 2, {}),                # 2-stage plan with a long K
    (2048, 2056, 200, SMALL, 2, {}),              # a coarser tile
    (4104, 4096, 520, BIG, 2, {"bias": "f16"}),   # 8 rows past a whole round
    (512, 40000, 264, BIG, 2, {"bias": "f32"}),   # columns cut off
    (4200, 4200, 328, BIG, 2, {"persistent": True, "num_ctas": 256}),
    (4200, 4200, 328, BIG, 2, {"c_f32": True}),
    (700, 1504, 2048, BIG, 2, {"c_f32": True}),   # planned: prior C in the loop
    (3072, 3072, 1280, MID, 3, {"c_f32": True}),  # large grids of small tiles
    (2048, 2048, 2048, SMALL, 3, {"c_f32": True}),
    # split-K: 3 stages for 2, and 128x128 tiles on the 16x16x32 loop (splits of
    # unequal length, a partial last k-tile, fewer rows than a wave tile)
    (300, 520, 5000, (128, 64, 64), 2, {"split_k": 4, "bias": "f16"}),
    (300, 520, 5000, MID, 2, {"split_k": 4, "bias": "f16", "activation": "relu"}),
    (129, 136, 9224, MID, 3, {"split_k": 16}),
    (7, 1032, 4096, MID, 2, {"split_k": 7, "c_f32": True}),
    (1000, 776, 4168, MID, 2, {"split_k": 4, "c_f32": True, "module_attrs": ATOMIC}),
    (129, 8, 9000, MID, 4, {"split_k": 3, "c_f32": True, "module_attrs": ATOMIC}),
]


@pytest.mark.parametrize("M,N,K,block,stages,options", CASES,
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else None)
def test_matches_planned_kernel(M, N, K, block, stages, options, device):
    print(f"grid split {M}x{N}x{K} {block} {options}", flush=True)
    w = configs.Workload("w", M, N, K, 0, configs.NORMAL, block, num_waves=4, stages=stages,
                         exact_tile=False, **options)
    plan = tb.plan_from_mlir(w.mlir())
    exact = tb.GemmDesc.from_config(plan.config)
    assert exact.kernel_name == plan.kernel_name
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
