"""GPU: tde_reduce_rms with a staged algorithm is one launch that also stores (or reads) the stage.  What it leaves in every
buffer must be what its two phases, called one at a time, leave there; a stage that overlaps an output is still correct."""
import pytest
import torch

from oracle import eager
from torch_dist_ext_amd import _capi

from helpers import bits_equal, run_hip

pytestmark = pytest.mark.gpu


# rows around a window of the owned-rows order (1024 * N), around one compute unit's share of packed rows, and fewer rows
# than ranks; row lengths of one wavefront, of less, and of several vectors per thread
@pytest.mark.parametrize("n,rank,tokens,hidden,dtype,quant,vpt,rpb", [
    (2, 0, 2047, 128, torch.bfloat16, "fp8_group", 0, 0), (2, 1, 2049, 128, torch.float32, "none", 0, 4),
    (4, 3, 4096, 64, torch.float16, "fp8_token", 1, 3), (4, 0, 4099, 72, torch.bfloat16, "none", 2, 2),
    (8, 7, 8191, 32, torch.float32, "fp8_static", 4, 0), (8, 3, 8200, 8, torch.bfloat16, "int8_token", 0, 0),
    (8, 6, 5, 1000, torch.float16, "int8_token", 4, 1), (8, 1, 300, 8192, torch.bfloat16, "fp8_token", 0, 0),
    (4, 2, 4097, 6, torch.float64, "none", 0, 0), (2, 1, 130, 2048, torch.float64, "none", 0, 0),
    # the norm phase alone takes other vectors per thread than the one launch: doubles one against four, four against one
    (2, 0, 300, 512, torch.float64, "none", 0, 0), (2, 1, 1400, 1960, torch.float64, "none", 0, 0), (4, 1, 3100, 1602, torch.float64, "none", 0, 0),
    # rows that are not whole 128-byte lines, T-typed rows beside the codes: owned rows four, their norm phase alone one
    (4, 1, 2100, 2820, torch.float32, "fp8_token", 0, 0),
])
def test_one_launch_equals_its_phases(cuda_device, n, rank, tokens, hidden, dtype, quant, vpt, rpb):
    print("case", n, rank, tokens, hidden, dtype, quant, vpt, rpb, flush=True)
    p, r, g = eager.make_inputs(n, tokens, hidden, dtype, 1.0, seed=700 + n)
    stage = torch.randn((tokens, hidden), generator=torch.Generator().manual_seed(7), dtype=torch.float64).to(dtype)
    stage[0, 0] = -0.0   # a delivered sum is taken as it is, sign of zero included
    kw = dict(rank=rank, stage_init=stage, vecs_per_thread=vpt, rows_per_block=rpb,
              static_scale=0.03 if quant == "fp8_static" else 0.0)
    for algo in (_capi.ALGO_STAGED, _capi.ALGO_STAGED_OWNED):
        one = run_hip(p, r, g, 1e-6, quant, algo=algo, **kw)
        two = run_hip(p, r, g, 1e-6, quant, algo=algo, calls=[(("reduce",), rank), (("norm",), rank)], **kw)
        for k in two:
            assert bits_equal(one[k], two[k]), (algo, k)


@pytest.mark.parametrize("where", ["norm_out", "residual_out", "residual_in"])
def test_stage_that_overlaps_another_buffer(cuda_device, where):
    """Both phases then still run one after the other: the residual is read, and an output written, after all the sums."""
    import torch_dist_ext_amd as tde
    print("case", where, flush=True)
    p, r, g = eager.make_inputs(4, 70, 1024, torch.bfloat16, 1.0, seed=9)
    want = eager.reduce_rms(p, p.float().sum(0).to(p.dtype) if where == "residual_in" else r, g, 1e-6, "none")
    parts = [p[i].to(cuda_device) for i in range(4)]
    buf = {"residual_in": r.to(cuda_device), "residual_out": torch.empty_like(r, device=cuda_device),
           "norm_out": torch.empty_like(r, device=cuda_device)}
    tde.reduce_rms_local_impl(parts, buf["residual_in"], g.to(cuda_device), buf["residual_out"], buf["norm_out"], None, None,
                              1e-6, tde.QUANT_NONE, tde.ALGO_STAGED, buf[where], 0.0)
    torch.cuda.synchronize()
    assert bits_equal(buf["residual_out"].cpu(), want["residual_out"])
    assert bits_equal(buf["norm_out"].cpu(), want["norm_out"])


@pytest.mark.parametrize("where", ["residual_ahead", "residual_behind", "gamma"])
@pytest.mark.parametrize("algo", [_capi.ALGO_STAGED, _capi.ALGO_STAGED_OWNED])
def test_stage_over_an_input_of_the_norm(cuda_device, where, algo):
    """What the norm reads through an overlap are sums of other rows, all of them stored before: the residual of row t is the stage's
    row t + 40 or t - 40, or gamma is the stage's last row.  A single launch would read most of them before they are there."""
    import torch_dist_ext_amd as tde
    print("case", where, algo, flush=True)
    shift, tokens, hidden, n = 40, 3000, 1024, 4
    p, r, g = eager.make_inputs(n, tokens, hidden, torch.bfloat16, 0.25, seed=11)
    sums = torch.zeros((tokens, hidden))
    for k in range(n):
        sums = sums + p[k].float()
    sums = sums.to(p.dtype)
    memory = torch.cat([r, r[:shift]]).to(cuda_device)
    before = memory.cpu()
    stage = memory[shift:] if where == "residual_behind" else memory[:tokens]
    if algo == _capi.ALGO_STAGED_OWNED:   # what the peers delivered, and nothing yet in this rank's rows (0, 4, 8, ...)
        owned = torch.arange(tokens) % n == 0
        stage.copy_(torch.where(owned[:, None], stage.cpu(), sums))
        before = memory.cpu()
    at = shift if where == "residual_behind" else 0
    before[at: at + tokens] = sums        # the memory once every sum has been stored
    res, gamma = r.to(cuda_device), g.to(cuda_device)
    if where == "gamma":
        gamma = stage[tokens - 4]         # an owned row
        want = eager.reduce_rms(p, r, sums[tokens - 4], 1e-6, "none")
    else:
        first = 0 if where == "residual_behind" else shift
        res = memory[first: first + tokens]
        want = eager.reduce_rms(p, before[first: first + tokens], g, 1e-6, "none")
    res_out, norm_out = torch.empty_like(r, device=cuda_device), torch.empty_like(r, device=cuda_device)
    tde.reduce_rms_local_impl([p[k].to(cuda_device) for k in range(n)], res, gamma, res_out, norm_out, None, None, 1e-6,
                              tde.QUANT_NONE, algo, stage, 0.0)
    torch.cuda.synchronize()
    assert bits_equal(res_out.cpu(), want["residual_out"])
    assert bits_equal(norm_out.cpu(), want["norm_out"])


@pytest.mark.parametrize("out", ["norm_out", "residual_out", "q_out"])
@pytest.mark.parametrize("algo", [_capi.ALGO_STAGED, _capi.ALGO_STAGED_OWNED])
def test_output_that_overlaps_a_partial(cuda_device, out, algo):
    """A caller may reuse the partials' memory for the outputs, shifted: no output is written before the last sum is stored."""
    import torch_dist_ext_amd as tde
    print("case", out, algo, flush=True)
    shift, tokens, hidden = 40, 3000, 1024
    p, r, g = eager.make_inputs(4, tokens, hidden, torch.bfloat16, 1.0, seed=10)
    want = eager.reduce_rms(p, r, g, 1e-6, "fp8_token")
    stage = p.float().sum(0).to(p.dtype).to(cuda_device)   # owned rows: what the peers delivered
    memory = torch.empty((tokens + shift, hidden), dtype=p.dtype, device=cuda_device)
    parts = [p[0].to(cuda_device), memory[shift:].copy_(p[1]), p[2].to(cuda_device), p[3].to(cuda_device)]
    buf = {k: torch.empty_like(r, device=cuda_device) for k in ("norm_out", "residual_out")}
    buf["q_out"] = torch.empty((tokens, hidden), dtype=torch.float8_e4m3fn, device=cuda_device)
    buf[out] = memory.view(torch.float8_e4m3fn).view(-1)[: tokens * hidden].view(tokens, hidden) if out == "q_out" else memory[:tokens]
    if out == "q_out":
        parts[1] = memory.view(-1)[: tokens * hidden].view(tokens, hidden).copy_(p[1])   # codes of row t lie on row t / 2
    scale = torch.empty(tokens, device=cuda_device)
    tde.reduce_rms_local_impl(parts, r.to(cuda_device), g.to(cuda_device), buf["residual_out"], buf["norm_out"], buf["q_out"], scale,
                              1e-6, tde.QUANT_FP8_TOKEN, algo, stage, 0.0)
    torch.cuda.synchronize()
    for got, name in ((buf["residual_out"], "residual_out"), (buf["norm_out"], "norm_out"), (buf["q_out"], "q"), (scale, "scale")):
        assert bits_equal(got.cpu(), want[name]), name
