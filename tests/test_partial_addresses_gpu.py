"""GPU: the partials' addresses reach the kernels as arguments, through the device pointer table, or some one way and some the
other; every mixture gives the same bits, in the fused launch and in the staged ones (which take the table separately)."""
import pytest
import torch

from oracle import eager
from torch_dist_ext_amd import _capi

from helpers import bits_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("known", ["", "0", "3", "02", "123", "0123"])
@pytest.mark.parametrize("algo", [_capi.ALGO_FUSED, _capi.ALGO_STAGED, _capi.ALGO_STAGED_OWNED])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float64])
def test_any_mixture_of_arguments_and_table(cuda_device, known, algo, dtype):
    print("case", known, algo, dtype, flush=True)
    n, tokens, hidden, rank, eps = 4, 37, 512, 1, 1e-6
    p, r, g = eager.make_inputs(n, tokens, hidden, dtype, 1.0, seed=5)
    want = eager.reduce_rms(p, r, g, eps, "none")
    parts = [p[k].to(cuda_device) for k in range(n)]
    res, gamma = r.to(cuda_device), g.to(cuda_device)
    res_out, norm_out, stage = (torch.full_like(res, float("nan")) for _ in range(3))
    if algo == _capi.ALGO_STAGED_OWNED:   # the peers' rows, each the sum in rank order
        acc = torch.zeros_like(p[0], dtype=torch.float64 if dtype == torch.float64 else torch.float32)
        for k in range(n):
            acc = acc + p[k]
        stage.copy_(acc.to(dtype))
        stage[rank::n] = float("nan")
    table = torch.tensor([t.data_ptr() if str(k) not in known else 0 for k, t in enumerate(parts)], dtype=torch.int64, device=cuda_device)
    prob = _capi.make_problem({torch.bfloat16: _capi.BF16, torch.float64: _capi.F64}[dtype], n, tokens, hidden, eps, algo=algo, rank=rank)
    _capi.reduce_rms(prob, [t.data_ptr() if str(k) in known else None for k, t in enumerate(parts)], res.data_ptr(),
                     res_out.data_ptr(), gamma.data_ptr(), norm_out=norm_out.data_ptr(), stage=stage.data_ptr(),
                     partial_table=table.data_ptr(), stream=torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert bits_equal(res_out.cpu(), want["residual_out"]) and bits_equal(norm_out.cpu(), want["norm_out"])
