"""Limits on resident workgroups per compute unit where launches are shorter, or their rows, than those of test_abi_host.py: on both sides
of each range, and what such launches leave."""
import pytest
import torch

from helpers import bits_equal, run_hip
from oracle import eager
from torch_dist_ext_amd import _capi

BF16, F16, F32 = _capi.BF16, _capi.F16, _capi.F32
FP8, GROUP, INT8, STATIC, NONE = _capi.QUANT_FP8_TOKEN, _capi.QUANT_FP8_GROUP, _capi.QUANT_INT8_TOKEN, _capi.QUANT_FP8_STATIC, _capi.QUANT_NONE


@pytest.mark.parametrize("dtype,n,tokens,hidden,quant,wn,algo,limit", [
    # four partials, four vectors per thread, only codes of a dynamic scale to store: 16 to 30 workgroups per unit
    (BF16, 4, 4095, 7168, FP8, 0, _capi.ALGO_AUTO, 0), (BF16, 4, 4096, 7168, FP8, 0, _capi.ALGO_AUTO, 2), (F16, 4, 7679, 8192, INT8, 0, _capi.ALGO_AUTO, 2),
    (F16, 4, 7680, 8192, INT8, 0, _capi.ALGO_AUTO, 0), (F32, 4, 5000, 4096, GROUP, 0, _capi.ALGO_AUTO, 2), (BF16, 4, 5000, 7168, FP8, 1, _capi.ALGO_AUTO, 0),
    (BF16, 4, 5000, 7168, STATIC, 0, _capi.ALGO_AUTO, 0), (BF16, 4, 5000, 7168, NONE, 0, _capi.ALGO_AUTO, 0), (BF16, 2, 5000, 7168, FP8, 0, _capi.ALGO_AUTO, 0),
    (BF16, 4, 5000, 4096, FP8, 0, _capi.ALGO_AUTO, 0),
    # short rows with a stage: six workgroups, of rows up to 181 vectors, in launches of 56 MB on
    (F16, 4, 26425, 1144, INT8, 0, _capi.ALGO_STAGED, 6), (F32, 4, 27056, 316, INT8, 0, _capi.ALGO_STAGED, 6), (BF16, 4, 9000, 1440, FP8, 0, _capi.ALGO_STAGED, 6),
    (BF16, 4, 9000, 1456, FP8, 0, _capi.ALGO_STAGED, 4), (BF16, 4, 9000, 1440, NONE, 0, _capi.ALGO_STAGED, 4), (BF16, 4, 8600, 520, FP8, 0, _capi.ALGO_STAGED, 4),
    (BF16, 8, 9000, 1440, FP8, 0, _capi.ALGO_STAGED, 4),
    # eight partials, rows of three wavefronts, and of four with T-typed output: 96 KiB from 48 workgroups per unit on
    (BF16, 8, 12287, 1280, FP8, 0, _capi.ALGO_AUTO, 6), (BF16, 8, 12288, 1280, FP8, 0, _capi.ALGO_AUTO, 4), (BF16, 8, 12288, 1544, FP8, 0, _capi.ALGO_AUTO, 5),
    (F32, 8, 12288, 772, NONE, 0, _capi.ALGO_AUTO, 4), (F16, 8, 12288, 1920, NONE, 0, _capi.ALGO_AUTO, 3), (F16, 8, 12287, 1920, NONE, 0, _capi.ALGO_AUTO, 4),
    (F16, 8, 12288, 2056, NONE, 0, _capi.ALGO_AUTO, 4), (F16, 8, 12288, 1024, NONE, 0, _capi.ALGO_AUTO, 4),
])
def test_limits(dtype, n, tokens, hidden, quant, wn, algo, limit):
    if torch.cuda.is_available() and _capi.device_info().compute_units != 256:
        pytest.skip("the row counts are for 256 compute units")
    p = _capi.make_problem(dtype, n, tokens, hidden, 1e-5, quant=quant, algo=algo, write_norm=wn, static_scale=0.5 if quant == STATIC else 0.0)
    assert _capi.plan(p).workgroups_per_cu == limit


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,n,tokens,hidden,quant,algo", [(torch.float16, 4, 4099, 6152, "int8_token", _capi.ALGO_AUTO), (torch.float32, 4, 8003, 400, "fp8_token", _capi.ALGO_STAGED),
                                                              (torch.float16, 8, 1027, 6200, "fp8_token", _capi.ALGO_AUTO),
                                                              (torch.bfloat16, 8, 12290, 1032, "none", _capi.ALGO_AUTO)])
def test_limited_launch_equals_the_unlimited(cuda_device, dtype, n, tokens, hidden, quant, algo):
    print("case", dtype, n, tokens, hidden, quant, algo, flush=True)
    p, r, g = eager.make_inputs(n, tokens, hidden, dtype, 1.0, seed=hidden)
    want = run_hip(p, r, g, 1e-6, quant, algo=algo, workgroups_per_cu=-1)
    got = run_hip(p, r, g, 1e-6, quant, algo=algo)
    for k in want:
        assert bits_equal(got[k], want[k]), k


@pytest.mark.parametrize("dtype,n,tokens,hidden,quant,wn,limit", [
    # fp16, two partials, codes beside the stage, four vectors per thread: two workgroups from 24 per unit on
    (F16, 2, 6143, 8192, FP8, 0, 0), (F16, 2, 6144, 8192, FP8, 0, 2), (F16, 2, 20000, 7424, STATIC, 1, 2), (F16, 2, 9000, 7680, GROUP, 0, 2), (F16, 2, 9000, 8184, INT8, 1, 2),
    (F16, 2, 9000, 8192, NONE, 0, 0), (BF16, 2, 9000, 8192, FP8, 0, 0), (F16, 2, 9000, 4096, FP8, 0, 0),
])
def test_staged_fp16_limits(dtype, n, tokens, hidden, quant, wn, limit):
    test_limits(dtype, n, tokens, hidden, quant, wn, _capi.ALGO_STAGED, limit)


@pytest.mark.gpu
def test_staged_fp16_limited_launch_equals_the_unlimited(cuda_device):
    test_limited_launch_equals_the_unlimited(cuda_device, torch.float16, 2, 6147, 7176, "int8_token", _capi.ALGO_STAGED)


@pytest.mark.parametrize("tokens,quant,wn,padded", [
    # eight partials, only codes of a dynamic scale to store, 16 to 24 workgroups per unit: the kernel for three wavefronts per SIMD with two workgroups by
    # its LDS; otherwise the one for two wavefronts, whose registers admit two, up to 24
    (4095, FP8, 0, False), (4096, FP8, 0, True), (6143, FP8, 0, True), (6144, FP8, 0, True), (4096, FP8, 1, False), (6143, NONE, 0, False), (6143, STATIC, 0, False),
    (6144, NONE, 0, True),
])
def test_two_workgroups_of_eight_partials(tokens, quant, wn, padded):
    if torch.cuda.is_available() and _capi.device_info().compute_units != 256:
        pytest.skip("the row counts are for 256 compute units")
    p = _capi.plan(_capi.make_problem(BF16, 8, tokens, 8192, 1e-5, quant=quant, write_norm=wn, static_scale=0.5 if quant == STATIC else 0.0))
    assert (p.workgroups_per_cu, p.lds_bytes) == (2, 80896 if padded else 36864)
