"""launch() looks at plain contiguous operands on a short path; everything
else goes to check_operands. Whatever check_operands refuses, launch refuses,
and operands it accepts give the same C either way."""
import pytest
import torch

import mini_triton_nvgpu_v1_amd as tb
from mini_triton_nvgpu_v1_amd import configs

pytestmark = pytest.mark.gpu

M, N, K = 64, 64, 32


def _shrunk(x):
    x = x.clone()
    x.untyped_storage().resize_(x.numel() * x.element_size() - 2)
    return x


BAD = {
    "dtype": lambda t: dict(t, a=t["a"].float()),
    "c_dtype": lambda t: dict(t, c=t["c"].float()),
    "transposed": lambda t: dict(t, b=torch.empty(N, K, dtype=torch.float16,
                                                  device=t["b"].device).t()),
    "short_rows": lambda t: dict(t, a=t["a"][:M - 1]),
    "short_flat": lambda t: dict(t, a=t["a"].reshape(-1)[8:]),
    "shrunk_storage": lambda t: dict(t, c=_shrunk(t["c"])),
    "host": lambda t: dict(t, b=t["b"].cpu()),
    "bias_dtype": lambda t: dict(t, bias=t["bias"].float()),
    "bias_short": lambda t: dict(t, bias=t["bias"][:N - 8].clone()),
}
GOOD = {
    "plain": lambda t: t,
    "flat": lambda t: dict(t, a=t["a"].reshape(-1)),          # not 2-D: footprint only
    "more_rows": lambda t: dict(t, a=torch.cat([t["a"], t["a"]])),
    "inside_storage": lambda t: dict(t, b=torch.cat([t["b"], t["b"]])[K:]),
    "parameter": lambda t: dict(t, b=torch.nn.Parameter(t["b"])),
}


@pytest.fixture()
def operands(device):
    g = torch.Generator(device=device).manual_seed(1)
    t = {"a": torch.randn(M, K, generator=g, device=device).half(),
         "b": torch.randn(K, N, generator=g, device=device).half(),
         "c": torch.empty(M, N, device=device, dtype=torch.float16),
         "bias": torch.randn(N, generator=g, device=device).half()}
    w = configs.Workload("w", M, N, K, 0, configs.NORMAL, (64, 64, 32), num_waves=4, bias="f16")
    return tb.plan_from_mlir(w.mlir()), t


@pytest.mark.parametrize("how", BAD)
def test_refused(how, operands):
    desc, t = operands
    bad = BAD[how](t)
    with pytest.raises(tb.TbError):
        desc.check_operands(bad["a"], bad["b"], bad["c"], None, bad["bias"])
    for launch in (desc.launch, desc.launch_noalloc):
        with pytest.raises(tb.TbError):
            launch(bad["a"], bad["b"], bad["c"], bias=bad["bias"])


@pytest.mark.parametrize("how", GOOD)
def test_accepted(how, operands):
    desc, t = operands
    ref = (t["a"].double() @ t["b"].double() + t["bias"].double())
    good = GOOD[how](t)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):  # the current stream is torch's
        desc.launch(good["a"], good["b"], good["c"], bias=good["bias"])
    torch.cuda.current_stream().wait_stream(stream)
    # f16 rounding of the result, 2^-11 of it, over the f32 sums' error
    assert ((good["c"].double() - ref).abs() <= 2.0 ** -10 * (ref.abs() + 1)).all()


def test_missing_bias(operands):
    desc, t = operands
    with pytest.raises(tb.TbError):
        desc.launch(t["a"], t["b"], t["c"])


def test_closed(operands):
    desc, t = operands
    desc.launch(t["a"], t["b"], t["c"], bias=t["bias"])
    desc.close()
    with pytest.raises(tb.TbError):
        desc.launch(t["a"], t["b"], t["c"], bias=t["bias"])
