"""GPU: rows of doubles with one, two and four 16-byte vectors per thread give the same bits in every buffer, whichever
algorithm sums the partials, and those of the oracle."""
import pytest
import torch

from oracle import eager
from torch_dist_ext_amd import _capi

from helpers import bits_equal, check_against_oracle, run_hip

pytestmark = pytest.mark.gpu


# a row of one vector, of one wavefront's four vectors per lane and one vector more or less, of an odd vector count, the
# longest; rows packed several to a workgroup with the last one incomplete
@pytest.mark.parametrize("n,tokens,hidden,rpb", [
    (2, 5, 2, 0), (8, 300, 510, 0), (4, 33, 512, 3), (2, 33, 514, 0), (4, 1027, 1398, 0), (8, 259, 2048, 0), (2, 3, 2046, 1),
])
def test_doubles_vectors_per_thread(cuda_device, n, tokens, hidden, rpb):
    print("case", n, tokens, hidden, rpb, flush=True)
    p, r, g = eager.make_inputs(n, tokens, hidden, torch.float64, 1.0, seed=800 + n)
    want = eager.reduce_rms(p, r, g, 1e-6, "none")
    stage = torch.randn((tokens, hidden), generator=torch.Generator().manual_seed(8), dtype=torch.float64)
    for algo in (_capi.ALGO_AUTO, _capi.ALGO_STAGED, _capi.ALGO_STAGED_OWNED):
        kw = {} if algo == _capi.ALGO_AUTO else dict(stage_init=stage)
        one, two, four = (run_hip(p, r, g, 1e-6, "none", algo=algo, rank=1, vecs_per_thread=v, rows_per_block=rpb, **kw)
                          for v in (1, 2, 4))
        if algo != _capi.ALGO_STAGED_OWNED:
            check_against_oracle({k: four[k] for k in ("residual_out", "norm_out")}, want, "none", gamma=g, eps=1e-6)
        for k in one:
            assert bits_equal(one[k], two[k]) and bits_equal(one[k], four[k]), (algo, k)

