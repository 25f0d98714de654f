"""fp16 rows of long launches of four partials, converted instead of computed in mixed instructions: every output bit for bit what one vector per thread
leaves and, the multiplication rounded twice among them, what the oracle says.  Around 190 of the 640-element case's normed elements lie on an fp16
rounding boundary, where a product rounded once differs.  Rows in place and moved, fused and beside a stage, codes alone of rows of more than 832
vectors, both sides of the range where the launch converts."""
import pytest
import torch

from helpers import bits_equal, check_against_oracle, run_hip
from oracle import eager
from torch_dist_ext_amd import _capi

pytestmark = pytest.mark.gpu


CASES = [  # rows, elements of a row, quant, algorithm
    (12290, 640, "none", _capi.ALGO_AUTO), (8195, 1032, "none", _capi.ALGO_AUTO), (8191, 640, "none", _capi.ALGO_AUTO), (4098, 640, "none", _capi.ALGO_STAGED),
    (4743, 1032, "none", _capi.ALGO_STAGED), (12290, 640, "fp8_static", _capi.ALGO_AUTO), (12288, 1032, "int8_token", _capi.ALGO_AUTO),
    (12289, 1024, "fp8_group", _capi.ALGO_AUTO), (12288, 6664, "fp8_token", _capi.ALGO_AUTO), (12289, 6656, "int8_token", _capi.ALGO_AUTO),
]


@pytest.mark.parametrize("tokens,hidden,quant,algo", CASES)
def test_converted_rows(cuda_device, tokens, hidden, quant, algo):
    print("case", tokens, hidden, quant, algo, flush=True)
    p, r, g = eager.make_inputs(4, tokens, hidden, torch.float16, 1.0, seed=hidden)
    scale = 0.03 if quant == "fp8_static" else 0.0
    alone = hidden > 6000   # codes alone; shorter rows with T-typed rows beside them
    want = run_hip(p, r, g, 1e-6, quant, algo=algo, vecs_per_thread=1, static_scale=scale, write_norm=not alone)
    got = run_hip(p, r, g, 1e-6, quant, algo=algo, vecs_per_thread=4, rows_per_block=1, static_scale=scale, write_norm=not alone)
    for k in want:
        assert bits_equal(got[k], want[k]), k
    rows = list(range(0, tokens, max(1, tokens * hidden // 2_000_000)))
    oracle = eager.reduce_rms(p[:, rows], r[rows], g, 1e-6, quant, static_scale=scale or None)
    check_against_oracle({k: v[rows] for k, v in got.items() if k != "stage"}, oracle, quant, gamma=g, eps=1e-6)
