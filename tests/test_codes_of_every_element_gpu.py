"""GPU: the codes of every 2-byte element there is, infinities and NaN included, and of fp32 elements around the codes'
boundaries.  A row of ones with eps 0 has reciprocal RMS 1, so its normed row is gamma itself."""
import pytest
import torch

from oracle import eager

from helpers import equal_where_not_nan, run_hip

pytestmark = pytest.mark.gpu


def _rows(elements):
    """Calls' inputs: gamma holds the elements, 4096 a call."""
    for at in range(0, elements.numel(), 4096):
        g = elements[at: at + 4096]
        r = torch.ones((2, g.numel()), dtype=g.dtype)
        yield torch.zeros((2, 2, g.numel()), dtype=g.dtype), r, g


def _check(elements, quant, scale=0.0, codes_of_nan=True):
    for p, r, g in _rows(elements):
        want = eager.reduce_rms(p, r, g, 0.0, quant, static_scale=scale) if quant == "fp8_static" else eager.reduce_rms(p, r, g, 0.0, quant)
        got = run_hip(p, r, g, 0.0, quant, static_scale=scale)
        assert equal_where_not_nan(got["norm_out"], g.expand(2, -1).contiguous())
        if quant != "fp8_static":
            assert equal_where_not_nan(got["scale"], want["scale"])
        assert equal_where_not_nan(got["q"], want["q"], nan_codes=quant != "int8_token"), (quant, scale)


def _patterns(dtype):
    return torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype)


# divisors of every kind: a power of two, all ones and all but one bit of the mantissa, the ends of the range that has a fast
# quotient and beyond, ordinary ones
SCALES = [1.0, 0.02, 1.0 - 2.0 ** -24, 2.0 - 2.0 ** -22, 1.0 + 2.0 ** -23, 2.0 ** -60, 2.0 ** 60, 2.0 ** -61, 2.0 ** 61, 1e-38, 3e38, 3.1e-5]


@pytest.mark.parametrize("scale", SCALES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_static_scale_every_element(cuda_device, dtype, scale):
    print("case", dtype, scale, flush=True)
    _check(_patterns(dtype), "fp8_static", scale=float(torch.tensor(scale, dtype=torch.float32)))


@pytest.mark.parametrize("quant", ["fp8_token", "fp8_group", "int8_token"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_dynamic_scale_every_finite_element(cuda_device, dtype, quant):
    """Sorted by magnitude, so that a row's (or group's) elements lie within its codes' range, with both signs of each."""
    e = _patterns(dtype)
    e = e[torch.isfinite(e.float())]
    e = e[torch.argsort(e.float().abs(), stable=True)]
    for lift in (1.0, 37.0):    # as they are, and with one element that takes them down the codes' range
        f = e.clone()
        if lift != 1.0:
            f[127::128] = (f[127::128].float() * lift).clamp(-6e4, 6e4).to(dtype)
        f = f[: f.numel() // 128 * 128]
        print("case", dtype, quant, lift, flush=True)
        _check(f, quant)


@pytest.mark.parametrize("scale", SCALES)
def test_static_scale_fp32_elements(cuda_device, scale):
    """Every boundary between two codes times the scale, and its neighbours; infinities, NaN, the largest and the smallest."""
    codes = torch.arange(256, dtype=torch.uint8).view(torch.float8_e4m3fn).float()
    codes = codes[torch.isfinite(codes)].sort().values
    at = (torch.cat([codes, (codes[1:] + codes[:-1]) / 2]).double() * scale).float()
    inf = torch.full_like(at, float("inf"))
    up, down = torch.nextafter(at, inf), torch.nextafter(at, -inf)
    e = torch.cat([at, up, down, torch.nextafter(up, inf), torch.nextafter(down, -inf),
                   torch.tensor([float("inf"), -float("inf"), float("nan"), 3.4e38, -3.4e38, 1e-45, -1e-45, 0.0, -0.0])])
    e = torch.cat([e, e[: -e.numel() % 4]]) if e.numel() % 4 else e
    print("case fp32", scale, e.numel(), flush=True)
    _check(e, "fp8_static", scale=float(torch.tensor(scale, dtype=torch.float32)))
