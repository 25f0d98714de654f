"""Which kernel a launch takes (tde_plan_route): the launches that other tests mean for one of them do take it, whatever becomes of the rules, and the
ordinary quantized call (codes alone) and partials from a pointer table through each."""
import pytest
import torch

import test_converted_rows_gpu
import test_shifted_rows_gpu
from helpers import DTYPE_CODE, QUANT_CODE, bits_equal, check_against_oracle, run_hip
from oracle import eager
from torch_dist_ext_amd import _capi


def route(n, tokens, hidden, dtype, quant, algo=_capi.ALGO_AUTO, rank=0, write_norm=1, **tuned):
    if torch.cuda.is_available() and _capi.device_info().compute_units != 256:
        pytest.skip("the row counts are for 256 compute units")
    return _capi.route(_capi.make_problem(DTYPE_CODE[dtype], n, tokens, hidden, 1e-6, quant=QUANT_CODE[quant], algo=algo, write_norm=write_norm, rank=rank,
                                          static_scale=0.03 if quant == "fp8_static" else 0.0, **tuned))


def test_rejects_what_the_plan_rejects():
    with pytest.raises(_capi.TdeError) as err:
        route(3, 16, 1024, torch.bfloat16, "none")
    assert err.value.status == _capi.ENRANKS
    assert _capi.load().tde_plan_route(None, _capi.RouteOut()) == _capi.EINVAL


@pytest.mark.parametrize("n,tokens,nvec,dtype,quant,algo,rank", test_shifted_rows_gpu.CASES)
def test_moved_rows_are_moved(n, tokens, nvec, dtype, quant, algo, rank):
    hidden, piece = nvec * 16 // dtype.itemsize, -(-tokens // 9) // n * n
    for write_norm in (0, 1):
        kw = dict(algo=algo, rank=rank, write_norm=write_norm)
        moved = [route(n, tokens, hidden, dtype, quant, vecs_per_thread=v, **kw).moved_to_lines for v in (0, 1, 2, 4)]
        assert moved[0] and sum(map(bool, moved)) >= 3, moved
        assert route(n, piece, hidden, dtype, quant, **kw).moved_to_lines == 0


@pytest.mark.parametrize("tokens,hidden,quant,algo", test_converted_rows_gpu.CASES)
def test_converted_rows_are_converted(tokens, hidden, quant, algo):
    kw = dict(algo=algo, write_norm=hidden < 6000, vecs_per_thread=4, rows_per_block=1)
    r = route(4, tokens, hidden, torch.float16, quant, **kw)
    assert r.kernel == (_capi.KERNEL_ROWS if tokens == 8191 else _capi.KERNEL_LONG if hidden == 6656 else _capi.KERNEL_CONVERTED) # beyond each end
    assert bool(r.moved_to_lines) == (hidden % 64 != 0 and (4 + 2) * tokens * hidden // 8 >> 16 >= 56)


@pytest.mark.parametrize("n,tokens,hidden,dtype,quant,kw,kernel,lanes", [
    (4, 12290, 640, torch.float16, "int8_token", dict(write_norm=0, vecs_per_thread=4, rows_per_block=1), _capi.KERNEL_LONG, 64),
    (4, 12290, 1032, torch.float16, "fp8_token", dict(write_norm=0, vecs_per_thread=4, rows_per_block=1), _capi.KERNEL_LONG, 64),
    (4, 12290, 6664, torch.float16, "fp8_token", dict(write_norm=0), _capi.KERNEL_CONVERTED, 256),
    (8, 2048, 8192, torch.bfloat16, "fp8_token", dict(write_norm=0), _capi.KERNEL_WIDE, 256),
    (8, 4096, 8192, torch.bfloat16, "fp8_token", dict(write_norm=0), _capi.KERNEL_ROWS, 256),
    (2, 67, 128, torch.bfloat16, "none", {}, _capi.KERNEL_SHORT, 16), (2, 67, 136, torch.float16, "none", {}, _capi.KERNEL_SHORT, 32),
    (4, 67, 128, torch.float32, "fp8_group", {}, _capi.KERNEL_SHORT, 32), (2, 67, 264, torch.bfloat16, "none", {}, _capi.KERNEL_ROWS, 64),
    (2, 67, 64, torch.float64, "none", {}, _capi.KERNEL_ROWS, 64),
])
def test_kernels(n, tokens, hidden, dtype, quant, kw, kernel, lanes):
    r = route(n, tokens, hidden, dtype, quant, **kw)
    assert (r.kernel, r.lanes_per_row) == (kernel, lanes)


@pytest.mark.gpu
@pytest.mark.parametrize("n,tokens,nvec,dtype,quant,algo,rank", [c for c in test_shifted_rows_gpu.CASES if c[4] != "none"])
def test_codes_alone_of_moved_rows(cuda_device, n, tokens, nvec, dtype, quant, algo, rank):
    """The kernels without T-typed rows beside the codes, every vectors-per-thread, against those with them."""
    print("case", n, tokens, nvec, dtype, quant, algo, rank, flush=True)
    p, r, g = eager.make_inputs(n, tokens, nvec * 16 // dtype.itemsize, dtype, 1.0, seed=nvec)
    kw = dict(quant=quant, algo=algo, rank=rank, static_scale=0.03 if quant == "fp8_static" else 0.0,
              stage_init=eager.reduce_residual(p, torch.zeros_like(r)) if algo == _capi.ALGO_STAGED_OWNED else None)
    want = run_hip(p, r, g, 1e-6, vecs_per_thread=1, **kw)
    for v in (0, 1, 2, 4):
        got = run_hip(p, r, g, 1e-6, vecs_per_thread=v, write_norm=False, **kw)
        for k in got:
            assert bits_equal(got[k], want[k]), (v, k)


@pytest.mark.gpu
@pytest.mark.parametrize("n,tokens,hidden,dtype,quant,moved", [
    (2, 67, 120, torch.bfloat16, "fp8_token", False), (8, 4103, 256, torch.float16, "none", False), (4, 259, 100, torch.float32, "int8_token", False),
    (4, 2602, 2072, torch.bfloat16, "fp8_token", True), (8, 7346, 260, torch.float32, "none", True), (2, 3702, 2040, torch.float16, "int8_token", True),
    (4, 1400, 514, torch.float64, "none", True), (4, 8195, 1032, torch.float16, "none", True),
])
def test_partials_from_a_table(cuda_device, n, tokens, hidden, dtype, quant, moved):
    print("case", n, tokens, hidden, dtype, quant, flush=True)
    r = route(n, tokens, hidden, dtype, quant)
    assert bool(r.moved_to_lines) == moved and (r.kernel == _capi.KERNEL_SHORT) == (not moved)
    p, res, g = eager.make_inputs(n, tokens, hidden, dtype, 1.0, seed=hidden)
    want = run_hip(p, res, g, 1e-6, quant)
    for rank in (0, n - 1):
        got = run_hip(p, res, g, 1e-6, quant, use_table=True, rank=rank)
        for k in want:
            assert bits_equal(got[k], want[k]), (rank, k)
    rows = list(range(0, tokens, max(1, tokens // 200)))
    check_against_oracle({k: v[rows] for k, v in want.items()}, eager.reduce_rms(p[:, rows], res[rows], g, 1e-6, quant), quant, gamma=g, eps=1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("n,tokens,nvec,dtype,quant,write_norm,moved", [
    (2, 1, 1, torch.bfloat16, "none", True, False), (8, 67, 15, torch.bfloat16, "fp8_token", False, False), (4, 4103, 16, torch.float16, "int8_token", True, False),
    (2, 6, 17, torch.float32, "fp8_token", True, False), (4, 259, 31, torch.float32, "none", True, False), (8, 4097, 32, torch.bfloat16, "fp8_static", False, False),
    (2, 7201, 129, torch.bfloat16, "none", True, True), (2, 3702, 255, torch.float16, "int8_token", False, True), (4, 614, 1023, torch.float16, "fp8_static", True, True),
    (8, 1026, 1021, torch.bfloat16, "fp8_token", False, True), (2, 2124, 253, torch.float32, "fp8_token", False, True), (8, 7346, 65, torch.float32, "none", True, True),
])
def test_traffic_skeletons_of_short_and_moved_rows(cuda_device, n, tokens, nvec, dtype, quant, write_norm, moved):
    """As test_traffic_skeleton_touches_every_byte_once, where the launch it stands for moves its rows or lets them share a wavefront: its outputs are the
    exclusive-or of all input rows."""
    print("case", n, tokens, nvec, dtype, quant, flush=True)
    hidden = nvec * 16 // dtype.itemsize
    r = route(n, tokens, hidden, dtype, quant, write_norm=int(write_norm))
    assert bool(r.moved_to_lines) == moved and (r.kernel == _capi.KERNEL_SHORT) == (not moved)
    p, res, g = eager.make_inputs(n, tokens, hidden, dtype, 1.0, seed=nvec)
    words = lambda t: t.contiguous().view(torch.int32).reshape(tokens, -1, 4)
    x = words(res).clone()
    for k in range(n):
        x ^= words(p[k])
    codes = (x[..., 0] ^ x[..., 1] ^ x[..., 2] ^ x[..., 3]) if dtype == torch.float32 else torch.stack([x[..., 0] ^ x[..., 2], x[..., 1] ^ x[..., 3]], dim=-1)
    out = run_hip(p, res, g, 1e-6, quant, write_norm=write_norm, static_scale=0.03 if quant == "fp8_static" else 0.0, calls=[(("traffic",), 0)])
    assert torch.equal(words(out["residual_out"]), x)
    if write_norm or quant == "none":
        assert torch.equal(words(out["norm_out"]), x)
    if quant != "none":
        assert torch.equal(out["q"].contiguous().view(torch.uint8).view(torch.int32).reshape(codes.shape), codes)


@pytest.mark.parametrize("n,nvec,tokens,quant,algo,vpt,moved", [
    # a wavefront to a row with four vectors per thread, up to four partials: moved from 56 MB on; longer rows from 28
    (2, 217, 2999, "none", _capi.ALGO_AUTO, 4, False), (2, 217, 4227, "none", _capi.ALGO_AUTO, 4, False), (2, 217, 4230, "none", _capi.ALGO_AUTO, 4, True),
    (4, 255, 2390, "none", _capi.ALGO_STAGED, 4, False), (4, 255, 2400, "none", _capi.ALGO_STAGED, 4, True), (8, 217, 1000, "none", _capi.ALGO_AUTO, 4, True),
    (2, 259, 1800, "none", _capi.ALGO_AUTO, 4, True), (2, 217, 3000, "none", _capi.ALGO_AUTO, 2, True),
])
def test_where_moving_begins(n, nvec, tokens, quant, algo, vpt, moved):
    assert bool(route(n, tokens, nvec * 8, torch.bfloat16, quant, algo=algo, vecs_per_thread=vpt).moved_to_lines) == moved
