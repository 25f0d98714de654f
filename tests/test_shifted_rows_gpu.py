"""Rows that start inside a line of memory, moved along their threads in long launches: what the launch leaves must be, bit for bit, what
short launches over pieces of the same rows leave, whose rows stay in place, and what the oracle says.  One vector more than whole
wavefronts and one less (the last vectors go to the first threads, or nearly do), every shift, one to four vectors per thread,
one and two rows to a workgroup, every form of the row kernel."""
import pytest
import torch

from helpers import bits_equal, check_against_oracle, run_hip
from oracle import eager
from torch_dist_ext_amd import _capi

CASES = [  # partials, rows, vectors of a row, dtype, quant, algorithm, rank
    (2, 7201, 129, torch.bfloat16, "none", _capi.ALGO_AUTO, 0),
    (2, 3702, 255, torch.float16, "int8_token", _capi.ALGO_AUTO, 0),
    (2, 1016, 1016, torch.bfloat16, "fp8_static", _capi.ALGO_AUTO, 0),
    (4, 2602, 259, torch.bfloat16, "fp8_token", _capi.ALGO_STAGED, 1),
    (4, 614, 1023, torch.float16, "fp8_static", _capi.ALGO_AUTO, 0),
    (8, 1030, 191, torch.bfloat16, "fp8_token", _capi.ALGO_AUTO, 0),
    (8, 1026, 1021, torch.bfloat16, "fp8_token", _capi.ALGO_AUTO, 0),
    (8, 2904, 327, torch.float16, "int8_token", _capi.ALGO_STAGED_OWNED, 5),
    (8, 7346, 65, torch.float32, "none", _capi.ALGO_AUTO, 0),
    (2, 2124, 253, torch.float32, "fp8_token", _capi.ALGO_AUTO, 0),
    (4, 1044, 515, torch.float32, "int8_token", _capi.ALGO_STAGED_OWNED, 2),
    (4, 1400, 257, torch.float64, "none", _capi.ALGO_AUTO, 0),
    (8, 514, 509, torch.float64, "none", _capi.ALGO_STAGED, 3),
    (2, 1230, 639, torch.float64, "none", _capi.ALGO_STAGED_OWNED, 1),
]


@pytest.mark.gpu
@pytest.mark.parametrize("n,tokens,nvec,dtype,quant,algo,rank", CASES)
def test_moved_rows_equal_rows_in_place(cuda_device, n, tokens, nvec, dtype, quant, algo, rank):
    print("case", n, tokens, nvec, dtype, quant, algo, rank, flush=True)
    scale = 0.03 if quant == "fp8_static" else 0.0
    p, r, g = eager.make_inputs(n, tokens, nvec * 16 // dtype.itemsize, dtype, 1.0, seed=nvec)
    kw = dict(quant=quant, algo=algo, rank=rank, static_scale=scale)
    stage = eager.reduce_residual(p, torch.zeros_like(r)) if algo == _capi.ALGO_STAGED_OWNED else None
    piece = -(-tokens // 9) // n * n  # owned rows keep their owner
    want = {}
    for a in range(0, tokens, piece):
        part = run_hip(p[:, a:a + piece], r[a:a + piece], g, 1e-6, stage_init=None if stage is None else stage[a:a + piece], **kw)
        for k, v in part.items():
            want.setdefault(k, []).append(v)
    want = {k: torch.cat(v) for k, v in want.items()}
    for v in (0, 1, 2, 4):
        got = run_hip(p, r, g, 1e-6, stage_init=stage, vecs_per_thread=v, **kw)
        for k in want:
            assert bits_equal(got[k], want[k]), (v, k)
    rows = list(range(34)) + [tokens - 2, tokens - 1]
    oracle = eager.reduce_rms(p[:, rows], r[rows], g, 1e-6, quant, static_scale=scale or None)
    check_against_oracle({k: v[rows] for k, v in got.items() if k != "stage"}, oracle, quant, gamma=g, eps=1e-6)


BF16, F16, F32 = _capi.BF16, _capi.F16, _capi.F32


@pytest.mark.parametrize("dtype,n,nvec,tokens,quant,algo,vpt", [
    # vectors per thread on both sides of each range: the launch's length, the row's, the number of rows
    (BF16, 8, 385, 9000, _capi.QUANT_FP8_TOKEN, _capi.ALGO_AUTO, 1), (BF16, 8, 383, 9000, _capi.QUANT_FP8_TOKEN, _capi.ALGO_AUTO, 2),
    (BF16, 8, 383, 8191, _capi.QUANT_FP8_TOKEN, _capi.ALGO_AUTO, 1), (F32, 8, 575, 8192, _capi.QUANT_NONE, _capi.ALGO_AUTO, 2),
    (BF16, 8, 601, 2048, _capi.QUANT_FP8_TOKEN, _capi.ALGO_AUTO, 4), (BF16, 8, 601, 2047, _capi.QUANT_FP8_TOKEN, _capi.ALGO_AUTO, 1),
    (F16, 2, 831, 2560, _capi.QUANT_INT8_TOKEN, _capi.ALGO_AUTO, 2), (F16, 2, 831, 2559, _capi.QUANT_INT8_TOKEN, _capi.ALGO_AUTO, 4),
    (F16, 2, 832, 2560, _capi.QUANT_INT8_TOKEN, _capi.ALGO_AUTO, 4), (F16, 2, 840, 2560, _capi.QUANT_INT8_TOKEN, _capi.ALGO_AUTO, 2),
    (BF16, 2, 901, 8192, _capi.QUANT_NONE, _capi.ALGO_AUTO, 1), (BF16, 2, 901, 8191, _capi.QUANT_NONE, _capi.ALGO_AUTO, 4),
    (BF16, 4, 901, 2048, _capi.QUANT_FP8_TOKEN, _capi.ALGO_AUTO, 2), (BF16, 4, 901, 2049, _capi.QUANT_FP8_TOKEN, _capi.ALGO_AUTO, 4),
    (BF16, 8, 521, 12000, _capi.QUANT_NONE, _capi.ALGO_STAGED_OWNED, 2), (BF16, 8, 521, 1199, _capi.QUANT_NONE, _capi.ALGO_STAGED_OWNED, 1),
    (BF16, 8, 520, 12000, _capi.QUANT_NONE, _capi.ALGO_STAGED_OWNED, 1),
])
def test_vectors_per_thread_of_moved_rows(dtype, n, nvec, tokens, quant, algo, vpt):
    if torch.cuda.is_available() and _capi.device_info().compute_units != 256:
        pytest.skip("the row counts are for 256 compute units")
    size = 4 if dtype == F32 else 2
    assert _capi.plan(_capi.make_problem(dtype, n, tokens, nvec * 16 // size, 1e-5, quant=quant, algo=algo)).vecs_per_thread == vpt
