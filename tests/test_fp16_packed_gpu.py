"""GPU: fp16 rows are added and multiplied in packed instructions that round once, where the eager composition rounds to fp32 and then to
fp16.  Every fp16 number goes through each of them: as a partial, as the residual and as gamma, beside numbers that put the result on
and beside rounding boundaries, subnormals, both zeros and infinities; in every geometry of the kernels."""
import pytest
import torch

from helpers import equal_where_not_nan, run_hip
from oracle import eager
from torch_dist_ext_amd import _capi

pytestmark = pytest.mark.gpu

EVERY = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(torch.float16)


@pytest.mark.parametrize("hidden,geometry", [(128, {}), (256, {}), (512, dict(vecs_per_thread=1)), (1024, dict(vecs_per_thread=2)), (2048, dict(vecs_per_thread=4)),
                                             (4096, dict(algo=_capi.ALGO_STAGED)), (4096, dict(algo=_capi.ALGO_STAGED_OWNED, rank=1))])
@pytest.mark.parametrize("n", [2, 4, 8])
def test_sums(cuda_device, n, hidden, geometry):
    print("case", n, hidden, geometry, flush=True)
    gen = torch.Generator().manual_seed(hidden + n)
    x = EVERY.view(-1, hidden)
    other = torch.randn(x.shape, generator=gen).half()
    # half a unit of the number beside it, a little more and a little less; the same number with the other sign; 0 and -0
    exponent = (x.view(torch.int16).int() >> 10) & 31
    half_unit = torch.ldexp(torch.ones(x.shape), (exponent.clamp(min=1) - 26)).half()
    for i, beside in enumerate([other, half_unit, half_unit * 1.5, -half_unit, -x, torch.zeros_like(x), torch.full_like(x, -0.0),
                                x[torch.randperm(x.shape[0], generator=gen)][:, torch.randperm(hidden, generator=gen)]]):
        p = torch.zeros((n, *x.shape), dtype=torch.float16)
        p[0], p[n - 1] = (x, beside) if i % 2 else (beside, x)
        if n > 2:
            p[1] = torch.randn(x.shape, generator=gen).half() * 1e-6
        for r in (torch.zeros_like(x), other, beside, x.flip(0)):
            stage = eager.reduce_residual(p, torch.full_like(x, -0.0)) if geometry.get("algo") == _capi.ALGO_STAGED_OWNED else None
            got = run_hip(p, r, torch.ones(hidden, dtype=torch.float16), 1e-6, stage_init=stage, **geometry)
            want = eager.reduce_residual(p, r)
            assert equal_where_not_nan(got["residual_out"], want), i


@pytest.mark.parametrize("hidden,geometry", [(128, {}), (256, {}), (512, dict(vecs_per_thread=1)), (4096, dict(vecs_per_thread=2)), (8192, dict(vecs_per_thread=4))])
@pytest.mark.parametrize("quant", ["fp8_token", "int8_token", "fp8_static"])
def test_products_and_codes(cuda_device, hidden, geometry, quant):
    finite = torch.where(EVERY.isfinite(), EVERY, torch.zeros_like(EVERY))
    scale = 0.03 if quant == "fp8_static" else 0.0
    gen = torch.Generator().manual_seed(hidden)
    for i, gamma in enumerate(finite[torch.randperm(65536, generator=gen)].view(-1, hidden)[:: max(1, 65536 // hidden // 16)]):
        print("case", hidden, quant, i, flush=True)
        p, r, _ = eager.make_inputs(2, 5, hidden, torch.float16, [1.0, 300.0, 1e-4][i % 3], seed=i)
        p[:, 3] *= 2e-5  # a row that reaches into the subnormal numbers
        r[3] *= 2e-5
        gamma = gamma if i % 2 else (gamma.float().clamp(-2, 2)).half()
        got = run_hip(p, r, gamma, 1e-6, quant, static_scale=scale, **geometry)
        want = eager.reduce_rms(p, r, gamma, 1e-6, quant, static_scale=scale or None)
        for k in want:
            undefined = ~want["norm_out"].isfinite().all(-1, keepdim=True) if k == "q" and quant == "int8_token" else None # infinity / infinity
            assert equal_where_not_nan(got[k], want[k], nan_codes=k == "q" and quant != "int8_token", ignore=undefined), k


@pytest.mark.parametrize("quant", ["none", "fp8_token", "fp8_group", "int8_token", "fp8_static"])
@pytest.mark.parametrize("hidden", [640, 1032])
def test_long_launches_keep_conversions(cuda_device, hidden, quant):
    """Four partials, four vectors per thread, 48 workgroups per compute unit: the kernels with conversions, rows in place and moved."""
    if quant == "fp8_group" and hidden % 128:
        pytest.skip("whole groups only")
    print("case", hidden, quant, flush=True)
    p, r, g = eager.make_inputs(4, 12290, hidden, torch.float16, 1.0, seed=hidden)
    kw = dict(quant=quant, static_scale=0.03 if quant == "fp8_static" else 0.0)
    want = run_hip(p, r, g, 1e-6, vecs_per_thread=1, **kw)
    for write_norm in (False, True):
        got = run_hip(p, r, g, 1e-6, vecs_per_thread=4, rows_per_block=1, write_norm=write_norm, **kw)
        for k in got:
            assert equal_where_not_nan(got[k], want[k]), k
