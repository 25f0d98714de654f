"""GPU: long launches of TDE_ALGO_STAGED are held to a few workgroups per compute unit; what they leave must be what the fused
launch and the sums leave.  Just from the launch length where the limit begins, two, three and four workgroups per unit, one
and two rows to a workgroup, a last workgroup that is not full."""
import pytest
import torch

from helpers import bits_equal
from torch_dist_ext_amd import _capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,tokens,hidden,dtype,mode,limit", [
    (8, 4096, 8192, torch.bfloat16, "fp8_token", 2), (8, 4095, 1032, torch.float16, "none", 0), (8, 4103, 1032, torch.float16, "int8_token", 4),
    (4, 8197, 520, torch.bfloat16, "fp8_static", 4), (4, 4100, 3008, torch.bfloat16, "fp8_token", 4), (4, 4200, 2048, torch.float32, "fp8_group", 3),
])
def test_long_staged_launch_equals_the_fused_one(cuda_device, n, tokens, hidden, dtype, mode, limit):
    import torch_dist_ext_amd as tde
    if _capi.device_info().compute_units == 256:
        code = {torch.bfloat16: _capi.BF16, torch.float16: _capi.F16, torch.float32: _capi.F32}[dtype]
        plan = _capi.plan(_capi.make_problem(code, n, tokens, hidden, 1e-6, quant=tde.QUANT_MODES[mode], algo=_capi.ALGO_STAGED,
                                             static_scale=0.03 if mode == "fp8_static" else 0.0))
        assert plan.workgroups_per_cu == limit
    print("case", n, tokens, hidden, dtype, mode, flush=True)
    g = torch.Generator(device=cuda_device).manual_seed(tokens)
    parts = [torch.randn((tokens, hidden), generator=g, device=cuda_device).to(dtype) for _ in range(n)]
    res = torch.randn((tokens, hidden), generator=g, device=cuda_device).to(dtype)
    gamma = (torch.rand(hidden, generator=g, device=cuda_device) + 0.5).to(dtype)
    scale = 0.03 if mode == "fp8_static" else 0.0
    stage = torch.full_like(res, float("nan"))
    want = tde.reduce_rms(parts, res, gamma, 1e-6, tde.QUANT_MODES[mode], static_scale=scale)
    for _ in range(2):
        got = tde.reduce_rms(parts, res, gamma, 1e-6, tde.QUANT_MODES[mode], algo=tde.ALGO_STAGED, stage=stage, static_scale=scale)
    assert got.keys() == want.keys()
    for k in want:
        assert bits_equal(got[k], want[k]), k
    sums = torch.zeros((tokens, hidden), device=cuda_device)
    for p in parts:
        sums = sums + p.float()
    assert bits_equal(stage, sums.to(dtype))
