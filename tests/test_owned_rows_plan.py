"""What tde_plan chooses for owned rows on both sides of each range of wavefronts per row, row counts and outputs."""
import pytest
import torch

from torch_dist_ext_amd import _capi

BF16, F16, F32 = _capi.BF16, _capi.F16, _capi.F32
NONE, FP8, INT8, STATIC = _capi.QUANT_NONE, _capi.QUANT_FP8_TOKEN, _capi.QUANT_INT8_TOKEN, _capi.QUANT_FP8_STATIC


def plan(dtype, n, nvec, tokens, quant, write_norm=0):
    if torch.cuda.is_available() and _capi.device_info().compute_units != 256:
        pytest.skip("the row counts are for 256 compute units; another number of units scales them")
    return _capi.plan(_capi.make_problem(dtype, n, tokens, nvec * 16 // (4 if dtype == F32 else 2), 1e-5, quant=quant, algo=_capi.ALGO_STAGED_OWNED,
                                         write_norm=write_norm, static_scale=0.5 if quant == STATIC else 0.0))


@pytest.mark.parametrize("dtype,nvec,tokens,quant,write_norm,vpt", [
    # T-typed output, rows inside lines of 5 to 8 wavefronts: one vector per thread from 4608 rows on, of 8 always
    (BF16, 261, 4607, NONE, 0, 2), (BF16, 261, 4608, NONE, 0, 1), (F16, 447, 4607, NONE, 0, 2), (F16, 447, 20000, NONE, 0, 1), (F32, 369, 17457, NONE, 0, 1),
    (BF16, 449, 2400, NONE, 0, 1), (F32, 511, 2400, NONE, 0, 1), (F16, 513, 20000, NONE, 0, 2), (F32, 639, 20000, NONE, 0, 2),
    # T-typed rows beside codes: of fp32 the same, of a 2-byte type eight wavefronts only
    (F32, 261, 4607, FP8, 1, 2), (F32, 261, 4608, FP8, 1, 1), (F32, 447, 9000, STATIC, 1, 1), (F32, 505, 3000, INT8, 1, 1), (F32, 513, 9000, INT8, 1, 2),
    (BF16, 261, 9000, STATIC, 1, 2), (F16, 505, 9000, INT8, 1, 1),
    # codes alone: two
    (F32, 369, 9000, FP8, 0, 2), (BF16, 505, 9000, STATIC, 0, 2), (F16, 261, 20000, INT8, 0, 2),
])
def test_vectors_per_thread_of_eight_partials(dtype, nvec, tokens, quant, write_norm, vpt):
    assert plan(dtype, 8, nvec, tokens, quant, write_norm).vecs_per_thread == vpt


@pytest.mark.parametrize("dtype,n,nvec,tokens,quant,write_norm,shared", [
    # up to four partials: few rows of a 2-byte type and more than 16 vectors have a wavefront each
    (BF16, 4, 17, 255, NONE, 0, False), (BF16, 4, 17, 256, NONE, 0, True), (F16, 2, 32, 1, INT8, 1, False), (BF16, 4, 16, 3, FP8, 0, True),
    (F32, 4, 30, 5, FP8, 0, True), (BF16, 8, 30, 5, FP8, 0, True),
    # two partials, many rows of more than 24 vectors whose T-typed rows are stored: from 30 MB on, T-typed output of fp32 from 72
    (BF16, 2, 25, 19660, NONE, 0, True), (BF16, 2, 25, 19661, NONE, 0, False), (F16, 2, 24, 40000, NONE, 0, True), (F16, 2, 32, 15360, STATIC, 1, False),
    (F16, 2, 32, 30000, INT8, 1, True), (BF16, 2, 32, 30000, FP8, 0, True), (F32, 2, 32, 36863, NONE, 0, True), (F32, 2, 32, 36864, NONE, 0, False),
    (F32, 2, 25, 19661, FP8, 1, False),
    (BF16, 4, 32, 30000, NONE, 0, True), (BF16, 8, 32, 30000, NONE, 0, True),
])
def test_rows_that_share_a_wavefront(dtype, n, nvec, tokens, quant, write_norm, shared):
    p = plan(dtype, n, nvec, tokens, quant, write_norm)
    assert (p.block_threads // p.rows_per_block < 64) == shared
