"""The vectors per thread that tde_plan chooses at the ends of each range of row lengths and row counts."""
import pytest
import torch

from torch_dist_ext_amd import _capi


def vecs(dtype, n, nvec, tokens, **kw):
    if torch.cuda.is_available() and _capi.device_info().compute_units != 256:
        pytest.skip("the row counts are for 256 compute units; another number of units scales them")
    size = {_capi.F64: 8, _capi.F32: 4}.get(dtype, 2)
    return _capi.plan(_capi.make_problem(dtype, n, tokens, nvec * 16 // size, 1e-5, **kw)).vecs_per_thread


@pytest.mark.parametrize("n,nvec,tokens,vpt", [
    (4, 1024, 255, 1), (4, 1024, 256, 4), (4, 1024, 3071, 4), (4, 1024, 3072, 1), (8, 1024, 6143, 4), (8, 1024, 6144, 1),
    (4, 768, 575, 4), (4, 768, 576, 1), (4, 767, 1535, 1), (8, 768, 6143, 4), (8, 768, 6144, 1), (8, 744, 1535, 4), (8, 745, 448, 1),
    (2, 768, 2303, 4), (2, 768, 2304, 1), (2, 767, 1024, 4), (2, 767, 1025, 1), (4, 769, 1536, 4), (4, 256, 256, 4), (4, 255, 256, 1),
    (2, 576, 1280, 4), (2, 576, 1281, 1), (4, 576, 1024, 4), (4, 576, 1025, 1), (8, 576, 1535, 4), (8, 575, 768, 1),
    (2, 577, 2303, 4), (2, 577, 2304, 1), (2, 584, 30000, 4), (2, 640, 30000, 4), (2, 641, 1024, 4), (2, 641, 1025, 1),
    (4, 648, 1535, 4), (4, 641, 576, 1), (2, 641, 1536, 1), (4, 830, 639, 4), (4, 830, 640, 1), (4, 830, 768, 4), (4, 832, 700, 4),
    (8, 320, 30000, 4), (8, 320, 1025, 1), (8, 321, 1536, 1), (2, 300, 640, 4), (2, 300, 641, 1), (2, 304, 1024, 4), (4, 300, 1280, 1),
    (4, 300, 1281, 4), (4, 300, 1537, 1), (4, 350, 1024, 4), (4, 350, 1216, 1), (4, 350, 1217, 4), (4, 352, 1280, 1),
    (4, 512, 1024, 4), (4, 512, 1280, 1), (4, 512, 1535, 4), (4, 512, 1536, 1), (2, 512, 1792, 1), (8, 512, 6143, 4),
    (2, 256, 2048, 4), (2, 256, 2049, 1), (8, 256, 1024, 4), (8, 256, 1025, 1), (8, 256, 2304, 4), (8, 256, 6144, 1),
    (2, 1000, 3071, 4), (2, 1001, 1280, 4), (2, 1001, 1281, 1), (4, 1001, 1152, 1), (4, 1017, 3071, 4), (8, 1001, 6143, 4),
    (8, 128, 8191, 1), (8, 128, 8192, 4), (8, 127, 8192, 1),
])
def test_doubles(n, nvec, tokens, vpt):
    assert vecs(_capi.F64, n, nvec, tokens) == vpt


NONE, FP8, GROUP, INT8, STATIC = (_capi.QUANT_NONE, _capi.QUANT_FP8_TOKEN, _capi.QUANT_FP8_GROUP, _capi.QUANT_INT8_TOKEN,
                                  _capi.QUANT_FP8_STATIC)


@pytest.mark.parametrize("dtype,n,nvec,tokens,quant,vpt", [
    # 13 wavefronts per row and more
    (_capi.BF16, 8, 768, 1000, FP8, 1), (_capi.BF16, 8, 769, 1000, FP8, 4), (_capi.BF16, 4, 830, 256, NONE, 1), (_capi.BF16, 4, 830, 257, NONE, 4),
    (_capi.BF16, 4, 830, 255, NONE, 2), (_capi.BF16, 4, 830, 4096, NONE, 4), (_capi.BF16, 4, 830, 4097, NONE, 1), (_capi.F16, 2, 830, 2048, INT8, 2), (_capi.F16, 2, 830, 2049, INT8, 4),
    (_capi.F16, 2, 830, 2049, NONE, 1), (_capi.F32, 2, 830, 2049, NONE, 4), (_capi.F16, 2, 896, 2049, NONE, 4),
    # ten wavefronts
    (_capi.BF16, 8, 577, 768, FP8, 2), (_capi.BF16, 8, 577, 1152, FP8, 1), (_capi.BF16, 8, 577, 16384, FP8, 1),
    (_capi.BF16, 4, 600, 16384, FP8, 2), (_capi.F32, 2, 600, 32768, NONE, 2), (_capi.BF16, 4, 600, 639, FP8, 1),
    (_capi.BF16, 4, 600, 1791, NONE, 2), (_capi.BF16, 4, 600, 1792, NONE, 1),
    # two partials, quantized
    (_capi.BF16, 2, 576, 1023, FP8, 1), (_capi.BF16, 2, 576, 1024, FP8, 2), (_capi.BF16, 2, 513, 4096, STATIC, 2),
    (_capi.BF16, 2, 528, 4095, GROUP, 1), (_capi.F16, 2, 641, 768, INT8, 2), (_capi.F16, 2, 768, 1536, INT8, 1),
    (_capi.F16, 2, 768, 2304, INT8, 2), (_capi.F32, 2, 768, 1536, INT8, 2), (_capi.BF16, 2, 384, 1536, FP8, 2),
    (_capi.BF16, 2, 449, 1536, FP8, 1), (_capi.BF16, 2, 320, 16383, FP8, 1), (_capi.F32, 2, 320, 1536, FP8, 2),
    (_capi.F32, 4, 513, 1536, FP8, 2), (_capi.BF16, 4, 513, 1536, FP8, 1),
    # T-typed output: the windows of row counts
    (_capi.BF16, 2, 641, 575, NONE, 1), (_capi.BF16, 2, 641, 576, NONE, 4), (_capi.BF16, 2, 768, 1280, NONE, 1),
    (_capi.BF16, 2, 512, 1536, NONE, 4), (_capi.BF16, 2, 512, 1537, NONE, 1), (_capi.BF16, 4, 512, 1023, NONE, 4), (_capi.BF16, 4, 512, 1024, NONE, 1),
    (_capi.F32, 2, 257, 1344, NONE, 4), (_capi.F32, 2, 256, 3071, NONE, 4), (_capi.F32, 4, 193, 2048, NONE, 4), (_capi.F32, 4, 193, 2049, NONE, 1),
    (_capi.F32, 4, 192, 2000, NONE, 1),
])
def test_row_lengths(dtype, n, nvec, tokens, quant, vpt):
    assert vecs(dtype, n, nvec, tokens, quant=quant, static_scale=0.5 if quant == STATIC else 0.0) == vpt


# Launches in which several vectors per thread measured slower than one: on both sides of each range, rows of whole 128-byte
# lines (a multiple of eight vectors) and others, with and without T-typed rows beside the codes.
@pytest.mark.parametrize("dtype,n,nvec,tokens,quant,wn,vpt", [
    # T-typed rows beside the codes, two partials
    (_capi.BF16, 2, 300, 20000, FP8, 0, 2), (_capi.BF16, 2, 300, 20000, FP8, 1, 1), (_capi.BF16, 2, 350, 3071, INT8, 1, 2),
    (_capi.BF16, 2, 350, 3072, INT8, 1, 1), (_capi.BF16, 2, 430, 1791, FP8, 1, 2), (_capi.BF16, 2, 430, 1792, FP8, 1, 1),
    (_capi.BF16, 2, 432, 8191, FP8, 1, 2), (_capi.BF16, 2, 432, 8192, FP8, 1, 1), (_capi.F32, 2, 430, 8191, FP8, 1, 2),
    (_capi.F32, 2, 430, 8192, FP8, 1, 1), (_capi.BF16, 2, 550, 1343, FP8, 1, 2), (_capi.BF16, 2, 550, 1600, FP8, 1, 1),
    (_capi.BF16, 2, 552, 1600, FP8, 1, 2), (_capi.BF16, 2, 550, 4096, STATIC, 0, 2), (_capi.BF16, 2, 550, 4096, STATIC, 1, 1),
    (_capi.F32, 2, 550, 4096, STATIC, 1, 2), (_capi.BF16, 2, 690, 1536, FP8, 1, 2), (_capi.BF16, 2, 690, 1537, FP8, 1, 1),
    (_capi.BF16, 2, 768, 1407, FP8, 1, 2), (_capi.BF16, 2, 768, 1408, FP8, 1, 1), (_capi.BF16, 2, 768, 20000, STATIC, 1, 1),
    (_capi.F32, 2, 740, 20000, STATIC, 1, 1), (_capi.F32, 2, 744, 20000, STATIC, 1, 2), (_capi.BF16, 2, 768, 1280, STATIC, 1, 2),
    (_capi.BF16, 2, 768, 1281, STATIC, 1, 1), (_capi.BF16, 2, 750, 1025, STATIC, 1, 1),
    # ten wavefronts
    (_capi.BF16, 2, 621, 8191, NONE, 0, 2), (_capi.BF16, 2, 621, 8192, NONE, 0, 1), (_capi.BF16, 2, 624, 8192, NONE, 0, 2),
    (_capi.F32, 2, 621, 12288, NONE, 0, 1), (_capi.BF16, 4, 621, 4095, STATIC, 0, 2), (_capi.BF16, 4, 621, 4096, STATIC, 0, 1),
    (_capi.BF16, 4, 621, 8191, FP8, 0, 1), (_capi.BF16, 4, 621, 8192, FP8, 0, 2), (_capi.BF16, 4, 624, 4096, FP8, 0, 2),
    (_capi.BF16, 4, 621, 1280, STATIC, 1, 2), (_capi.BF16, 4, 621, 1281, STATIC, 1, 1), (_capi.BF16, 4, 621, 1792, FP8, 1, 1),
    (_capi.BF16, 8, 600, 775, FP8, 0, 2), (_capi.BF16, 8, 600, 776, FP8, 0, 1), (_capi.BF16, 8, 600, 832, FP8, 0, 2),
    # 13 and 14 wavefronts
    (_capi.BF16, 8, 771, 768, STATIC, 0, 1), (_capi.BF16, 8, 771, 769, STATIC, 0, 4), (_capi.BF16, 8, 776, 641, STATIC, 0, 4),
    (_capi.BF16, 8, 801, 650, NONE, 0, 1), (_capi.BF16, 8, 801, 650, FP8, 0, 4), (_capi.F32, 4, 867, 640, NONE, 0, 4),
    (_capi.F32, 4, 867, 641, NONE, 0, 1), (_capi.F32, 4, 867, 769, NONE, 0, 4), (_capi.BF16, 4, 850, 448, STATIC, 0, 4),
    (_capi.BF16, 4, 850, 449, STATIC, 0, 1), (_capi.BF16, 4, 850, 800, STATIC, 1, 1), (_capi.BF16, 4, 850, 3072, STATIC, 1, 1),
    (_capi.BF16, 4, 848, 3072, STATIC, 1, 4), (_capi.F32, 4, 800, 383, GROUP, 0, 1), (_capi.F32, 4, 800, 384, GROUP, 0, 4),
    # one partial step of the launch
    (_capi.BF16, 2, 256, 2048, NONE, 0, 4), (_capi.BF16, 2, 256, 2049, NONE, 0, 1), (_capi.BF16, 2, 256, 2240, NONE, 0, 4),
    (_capi.BF16, 2, 576, 1343, FP8, 0, 2), (_capi.BF16, 2, 576, 1344, FP8, 0, 1), (_capi.BF16, 2, 576, 1537, FP8, 0, 2),
])
def test_rows_that_lost(dtype, n, nvec, tokens, quant, wn, vpt):
    assert vecs(dtype, n, nvec, tokens, quant=quant, write_norm=wn, static_scale=0.5 if quant == STATIC else 0.0) == vpt


@pytest.mark.parametrize("n,nvec,tokens,quant,vpt", [
    (2, 321, 1023, FP8, 1), (2, 321, 1024, FP8, 2), (2, 353, 5000, FP8, 1), (2, 448, 5000, FP8, 1), (4, 448, 1024, INT8, 2), (4, 512, 5000, FP8, 1),
    (8, 513, 2048, FP8, 2), (2, 576, 4096, FP8, 2), (8, 640, 5000, FP8, 2), (8, 768, 2048, FP8, 4), (2, 768, 4096, FP8, 2),
    (8, 700, 5000, NONE, 1),
])
def test_owned_row_lengths(n, nvec, tokens, quant, vpt):
    assert vecs(_capi.BF16, n, nvec, tokens, quant=quant, algo=_capi.ALGO_STAGED_OWNED) == vpt


# Rows of eleven and twelve wavefronts on two partials: two of them fit a compute unit, so from a little beyond two rows per unit
# several vectors per thread pay.
@pytest.mark.parametrize("dtype,nvec,tokens,quant,wn,vpt", [
    (_capi.BF16, 768, 543, FP8, 0, 1), (_capi.BF16, 768, 544, FP8, 0, 2), (_capi.F32, 641, 767, INT8, 1, 2), (_capi.BF16, 640, 544, FP8, 0, 1),
    (_capi.BF16, 768, 543, STATIC, 1, 1), (_capi.BF16, 768, 544, STATIC, 1, 4), (_capi.BF16, 768, 1279, STATIC, 1, 4), (_capi.BF16, 650, 1024, STATIC, 1, 4),
    (_capi.BF16, 650, 1025, STATIC, 1, 1), (_capi.BF16, 704, 767, GROUP, 1, 2), (_capi.F32, 704, 1200, GROUP, 1, 4), (_capi.BF16, 768, 600, STATIC, 0, 1),
])
def test_just_beyond_two_rows_per_unit(dtype, nvec, tokens, quant, wn, vpt):
    assert vecs(dtype, 2, nvec, tokens, quant=quant, write_norm=wn, static_scale=0.5 if quant == STATIC else 0.0) == vpt


# Beside T-typed rows of fp32, two vectors per thread with twelve wavefronts were slower than one at 590 to 700 rows; four are not.
@pytest.mark.parametrize("nvec,tokens,quant,wn,vpt", [
    (768, 543, FP8, 1, 1), (768, 544, FP8, 1, 4), (768, 640, INT8, 1, 4), (705, 640, FP8, 1, 4), (704, 640, FP8, 1, 2), (768, 767, FP8, 1, 4),
    (768, 768, FP8, 1, 2), (768, 640, FP8, 0, 2),
])
def test_twelve_wavefronts_beside_rows_of_fp32(nvec, tokens, quant, wn, vpt):
    assert vecs(_capi.F32, 2, nvec, tokens, quant=quant, write_norm=wn) == vpt
