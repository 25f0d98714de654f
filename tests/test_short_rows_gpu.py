"""GPU: rows of up to 32 vectors, two or four to a wavefront, against the oracle: slots of 16 and 32 lanes and the row lengths beside
them, no lane left over and one, every kind of remainder of the row sum, a last wavefront that is not full, whole and half workgroups,
owned rows around a window of their order."""
import pytest
import torch

from oracle import eager
from torch_dist_ext_amd import _capi

from helpers import bits_equal, check_against_oracle, equal_where_not_nan, run_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("quant", ["none", "fp8_token", "fp8_group", "int8_token", "fp8_static"])
def test_rows_that_share_a_wavefront(cuda_device, dtype, quant):
    vec = 16 // dtype.itemsize
    for i, nvec in enumerate([32] if quant == "fp8_group" and vec == 4 else [16, 32] if quant == "fp8_group" else [1, 2, 3, 9, 15, 16, 17, 21, 31, 32, 33]):
        for j, tokens in enumerate([1, 6, 67, 4103]):
            n = [2, 4, 8][(i + j) % 3]
            print("case", dtype, quant, n, tokens, nvec, flush=True)
            p, r, g = eager.make_inputs(n, tokens, nvec * vec, dtype, 1.0, seed=nvec)
            scale = 0.03 if quant == "fp8_static" else 0.0
            want = eager.reduce_rms(p, r, g, 1e-6, quant, static_scale=scale or None)
            for write_norm in (False, True):
                got = run_hip(p, r, g, 1e-6, quant, write_norm=write_norm, static_scale=scale)
                check_against_oracle(got, want, quant, gamma=g, eps=1e-6)


@pytest.mark.parametrize("n,rank,tokens,nvec,dtype", [
    (2, 1, 2047, 15, torch.bfloat16), (2, 0, 2050, 32, torch.float32), (4, 3, 4099, 16, torch.float16), (4, 1, 3, 31, torch.bfloat16),
    (8, 5, 8191, 17, torch.bfloat16), (8, 0, 8197, 5, torch.float32), (8, 7, 6, 24, torch.float16),
])
def test_staged_forms_equal_one_row_to_a_wavefront(cuda_device, n, rank, tokens, nvec, dtype):
    print("case", n, rank, tokens, nvec, dtype, flush=True)
    p, r, g = eager.make_inputs(n, tokens, nvec * 16 // dtype.itemsize, dtype, 1.0, seed=n)
    stage = torch.randn((tokens, g.numel()), generator=torch.Generator().manual_seed(7)).to(dtype)
    for algo in (_capi.ALGO_STAGED, _capi.ALGO_STAGED_OWNED):
        kw = dict(algo=algo, rank=rank, stage_init=stage)
        want = run_hip(p, r, g, 1e-6, "int8_token", vecs_per_thread=1, **kw)
        for calls in (None, [(("reduce",), rank), (("norm",), rank)]):
            got = run_hip(p, r, g, 1e-6, "int8_token", calls=calls, **kw)
            for k in want:
                assert bits_equal(got[k], want[k]), (algo, calls, k)


def test_one_row_that_is_not_finite_leaves_its_neighbours(cuda_device):
    """NaN, infinity and magnitudes outside the fast paths' ranges in one of the rows of a wavefront; an all-zero row without eps."""
    for nvec in (15, 30):
        for value in (float("nan"), float("inf"), 2.0 ** 70, 2.0 ** -70, 0.0):
            print("case", nvec, value, flush=True)
            p, r, g = eager.make_inputs(4, 9, nvec * 8, torch.bfloat16, 1.0, seed=3)
            if value == value and abs(value) != float("inf"):
                p[:, 5] *= value
                r[5] *= value
            else:
                p[1, 5, 7] = value
            rest = [i for i in range(9) if i != 5]
            got, want = run_hip(p, r, g, 0.0, "fp8_token"), eager.reduce_rms(p, r, g, 0.0, "fp8_token")
            alone = run_hip(p, r, g, 0.0, "fp8_token", vecs_per_thread=1)
            for k in want:
                assert bits_equal(got[k][rest], want[k][rest]), k
                assert equal_where_not_nan(got[k], alone[k], nan_codes=k == "q"), k
