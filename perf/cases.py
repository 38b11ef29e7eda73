"""The GEMM calls a program makes through this package, as measurable cases.

Each case is one tb.matmul configuration: a problem size, the tile and wave
count its module asks for, and the options used in earnest (f16 C = A*B, f32
C += A*B, bias / activation / clamp, split-K with either reduction, persistent
order). ``prepare`` runs the plan pipeline and makes the operands, ``run`` is
the launch.

The listed cases come from the package's own workloads (configs.py), the
fair benchmark's case list and the large ragged cases of the tests; the few
others are generic. ``draw`` gives sizes over the same ranges.
"""
import math

import torch

import mini_triton_nvgpu_v1_amd as tb
from mini_triton_nvgpu_v1_amd import configs


def _case(m, n, k, block, waves, stages=2, **options):
    bm, bn, bk = block
    case = {"m": m, "n": n, "k": k, "block_m": bm, "block_n": bn, "block_k": bk,
            "waves": waves, "stages": stages, "c": "f16", "bias": "", "act": "",
            "clamp": False, "split_k": 1, "atomic": False, "persistent": False,
            "noalloc": False, "batch": 1}
    case.update(options)
    return case


def listed():
    def named(name, *args, **kw):
        return dict(_case(*args, **kw), name=name)

    return [
        # the smallest workload: one tile, one k-tile, launched with the
        # operand checks a call with tensors makes
        named("smoke_64x64x32", 64, 64, 32, (64, 64, 32), 4),
        # the fair benchmark's largest ragged small case, f32 C += A*B, as a
        # batch of eight: tb.matmul has no batch dimension, so a program binds
        # one launcher per product and calls them in turn
        named("general_448x288x64_b8", 448, 288, 64, (64, 64, 64), 4, c="f32", batch=8),
        # a mid-sized layer whose sizes divide by no tile, K included, with
        # every fused step
        named("ragged_1000x1496x712_silu", 1000, 1496, 712, (256, 256, 64), 4,
              bias="f32", act="silu", clamp=True),
        # the ordinary square product on 128x128 tiles
        named("gemm_2048_tile128", 2048, 2048, 2048, (128, 128, 64), 4, 3),
        # few rows against a large weight matrix (decoding): split over K to
        # fill the card, no workspace of the caller's
        named("skinny_64x4096x4096_gelu", 64, 4096, 4096, (64, 128, 64), 4, 3, split_k=8,
              bias="f16", act="gelu_tanh", noalloc=True),
        # a small result with a long K, deterministic split-K
        named("splitk_512x512x16384", 512, 512, 16384, (128, 64, 64), 8, 3, split_k=8),
        # accumulating a weight gradient: f32 C += A*B over a long ragged K,
        # atomic split-K
        named("atomic_1024x1024x8200", 1024, 1024, 8200, (128, 128, 64), 4, 2, split_k=4,
              c="f32", atomic=True),
        # the headline GEMM
        named("gemm_4096", 4096, 4096, 4096, (256, 256, 64), 4),
        # the same as a layer: bias and GELU fused
        named("gemm_4096_bias_gelu", 4096, 4096, 4096, (256, 256, 64), 4, bias="f16",
              act="gelu_tanh"),
        # the same as the reference's f32 C += A*B
        named("gemm_4096_f32_accumulate", 4096, 4096, 4096, (256, 256, 64), 4, c="f32"),
        # a layer over a number of rows that is no multiple of anything, with a
        # ragged K (K % 64 = 8)
        named("ragged_5000x4096x4104", 5000, 4096, 4104, (256, 256, 64), 4),
        # the largest: persistent programs over 1024 tiles
        named("persistent_8192", 8192, 8192, 8192, (256, 256, 64), 4, persistent=True),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], uniform over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def _tiles(m, n, block):
    return -(-m // block[0]) * -(-n // block[1])


def draw(rng):
    kind = rng.choice(("small", "small_batch", "layer", "square", "skinny", "splitk",
                       "atomic", "large", "large_epilogue", "large_f32", "persistent"))
    if kind in ("small", "small_batch"):
        m, n, k = _log(rng, 1, 512), _log(rng, 8, 512, 8), _log(rng, 8, 256, 8)
        block = rng.choice(((64, 64, 32), (64, 64, 64), (128, 128, 32), (128, 128, 64)))
        return _case(m, n, k, block, 4, c=rng.choice(("f16", "f32")),
                     batch=8 if kind == "small_batch" else 1)
    if kind == "layer":
        m, n, k = _log(rng, 200, 2048), _log(rng, 512, 3072, 8), _log(rng, 256, 3072, 8)
        block, stages = rng.choice((((128, 128, 64), 3), ((256, 256, 64), 2)))
        return _case(m, n, k, block, 4, stages, bias=rng.choice(("f16", "f32")),
                     act=rng.choice(("relu", "gelu_tanh", "silu")), clamp=rng.random() < 0.5)
    if kind == "square":
        m, n, k = (_log(rng, 1000, 3000, 8) for _ in range(3))
        return _case(m, n, k, (128, 128, 64), 4, 3)
    if kind == "skinny":
        m, n, k = _log(rng, 1, 128), _log(rng, 1024, 8192, 8), _log(rng, 2048, 8192, 8)
        block = (64, 128, 64)
        split = max(2, min(16, 256 // _tiles(m, n, block)))
        return _case(m, n, k, block, 4, 3, split_k=split, bias=rng.choice(("", "f16")),
                     act=rng.choice(("", "gelu_tanh", "silu")), noalloc=rng.random() < 0.5)
    if kind in ("splitk", "atomic"):
        m, n, k = _log(rng, 200, 1100), _log(rng, 200, 1100, 8), _log(rng, 4096, 16384, 8)
        block, waves, stages = (((128, 64, 64), 8, 3) if kind == "splitk"
                                else ((128, 128, 64), 4, 2))
        split = max(2, min(16, 256 // _tiles(m, n, block)))
        if kind == "atomic":
            return _case(m, n, k, block, waves, stages, split_k=split, c="f32", atomic=True)
        return _case(m, n, k, block, waves, stages, split_k=split,
                     c=rng.choice(("f16", "f32")))
    block = (256, 256, 64)
    if kind == "persistent":
        m, n, k = (_log(rng, 4200, 8000, 8) for _ in range(3))
        return _case(m, n, k, block, 4, persistent=True)
    m, n, k = _log(rng, 2048, 5000), _log(rng, 2048, 5000, 8), _log(rng, 1024, 6000, 8)
    if kind == "large_f32":
        return _case(m, n, k, block, 4, c="f32")
    if kind == "large_epilogue":
        return _case(m, n, k, block, 4, bias=rng.choice(("f16", "f32")),
                     act=rng.choice(("relu", "gelu_tanh", "silu")))
    return _case(m, n, k, block, 4)


def _module(case):
    """The case's tb.matmul module."""
    block = (case["block_m"], case["block_n"], case["block_k"])
    m, n, k = case["m"], case["n"], case["k"]
    w = configs.Workload(
        "case", m, n, k, 0, configs.NORMAL, block, num_waves=case["waves"],
        stages=case["stages"], split_k=case["split_k"], persistent=case["persistent"],
        exact_tile=m % block[0] == 0 and n % block[1] == 0 and k % block[2] == 0,
        num_ctas=min(256, _tiles(m, n, block)) if case["persistent"] else 1,
        bias=case["bias"], activation=case["act"],
        clamp_min=-0.25 if case["clamp"] else None, clamp_max=2.0 if case["clamp"] else None,
        c_f32=case["c"] == "f32",
        module_attrs={"tb.reduction-mode": '"split_k_parallel"'} if case["atomic"] else {})
    return w.mlir()


def _inputs(case, seed):
    """Per product of the batch: A like activations, N(0, 1); B like weights,
    N(0, 1) / sqrt(K); the bias; and the prior C of a C += A*B."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    m, n, k = case["m"], case["n"], case["k"]

    def normal(*shape, scale=1.0, dtype=torch.float16):
        x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
        return (x * scale).to(dtype)

    out = []
    for _ in range(case["batch"]):
        a, b = normal(m, k), normal(k, n, scale=1.0 / math.sqrt(k))
        bias = None
        if case["bias"]:
            bias = normal(n, scale=0.5,
                          dtype=torch.float16 if case["bias"] == "f16" else torch.float32)
        c = (normal(m, n, dtype=torch.float32) if case["c"] == "f32"
             else torch.empty((m, n), dtype=torch.float16, device="cuda"))
        out.append((a, b, c, bias))
    return out


def prepare(case, seed):
    desc = tb.plan_from_mlir(_module(case))
    ops = _inputs(case, seed)
    noalloc = case["noalloc"] and desc.workspace_bytes <= tb.NOALLOC_SCRATCH_BYTES
    ws = None
    if desc.workspace_bytes and not noalloc:
        ws = torch.empty(desc.workspace_bytes, dtype=torch.uint8, device="cuda")
    state = {"desc": desc, "ops": ops, "ws": ws, "noalloc": noalloc, "bound": None}
    if case["batch"] > 1:
        state["bound"] = [desc.bind(a, b, c, ws, bias=bias) for a, b, c, bias in ops]
    return state


def run(state):
    if state["bound"] is not None:
        for launch in state["bound"]:
            launch()
        return [c for _, _, c, _ in state["ops"]]
    a, b, c, bias = state["ops"][0]
    if state["noalloc"]:
        state["desc"].launch_noalloc(a, b, c, bias=bias)
    else:
        state["desc"].launch(a, b, c, state["ws"], bias=bias)
    return c


def work(case):
    m, n, k = case["m"], case["n"], case["k"]
    c_bytes = 8 * m * n if case["c"] == "f32" else 2 * m * n  # f32 C: read and written
    bias = {"": 0, "f16": 2, "f32": 4}[case["bias"]] * n
    return {"bytes": case["batch"] * (2 * (m * k + k * n) + c_bytes + bias),
            "flops": case["batch"] * 2 * m * n * k}


def tolerance(case):
    # about four times the largest error against 64 bits over the ranges: f16
    # results 2.1e-4 of the norm and 4.9e-4 of a value (their rounding), f32
    # results 4.7e-7 and 3.7e-6
    if case["c"] == "f16":
        return {"rel": 8e-4, "max": 2e-3}
    return {"rel": 2e-6, "max": 1.5e-5}


def exact(case, seed):
    outs = []
    for a, b, c, bias in _inputs(case, seed):
        x = a.double() @ b.double()
        if case["c"] == "f32":
            x += c.double()
        if bias is not None:
            x += bias.double()
        if case["act"] == "relu":
            x = x.clamp_min(0)
        elif case["act"] == "gelu_tanh":
            x = 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))
        elif case["act"] == "silu":
            x = x * torch.sigmoid(x)
        if case["clamp"]:
            x = x.clamp(-0.25, 2.0)
        outs.append(x)
    return outs if case["batch"] > 1 else outs[0]
