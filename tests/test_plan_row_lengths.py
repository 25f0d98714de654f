"""The vectors per thread that tde_plan chooses at the ends of each range of row lengths and row counts."""
import pytest
import torch

from torch_dist_ext_amd import _capi


def vecs(dtype, n, nvec, tokens, **kw):
    if torch.cuda.is_available() and _capi.device_info().compute_units != 256:
        pytest.skip("expectations are for 256 compute units")
    size = {_capi.F64: 8, _capi.F32: 4}.get(dtype, 2)
    return _capi.plan(_capi.make_problem(dtype, n, tokens, nvec * 16 // size, 1e-5, **kw)).vecs_per_thread


@pytest.mark.parametrize("n,nvec,tokens,vpt", [
    (4, 1024, 255, 1), (4, 1024, 256, 4), (4, 1024, 3071, 4), (4, 1024, 3072, 1), (8, 1024, 6143, 4), (8, 1024, 6144, 1),
    (4, 768, 1536, 4), (4, 767, 1535, 4), (4, 767, 1536, 1), (4, 769, 1536, 4), (4, 256, 256, 4), (4, 255, 256, 1),
    (2, 576, 1536, 1), (2, 577, 30000, 4), (2, 640, 30000, 4), (2, 641, 1536, 1),
    (8, 320, 30000, 4), (8, 321, 1536, 1), (8, 128, 8191, 1), (8, 128, 8192, 4), (8, 127, 8192, 1),
])
def test_doubles(n, nvec, tokens, vpt):
    assert vecs(_capi.F64, n, nvec, tokens) == vpt
