"""The workloads whose speed is tracked: one rank's reduce + residual + RMSNorm (+ quant) stage as a program calls it.

Every case goes through the package's public entry points with its inputs already on the GPU:

  functional  allreduce_rms / allreduce_rms_quant: a model layer's call through the workspace table, outputs allocated
              by the operator
  in_place    allreduce_rms_fusion_impl / allreduce_rms_quant_fusion_impl: the same with the caller's own output buffers
  partials    reduce_rms: the partials as a list of tensors; also the way to the staged algorithms (the reference's
              two-shot structure: the sum of the partials in a stage buffer, then the norm over its rows)
"""
import math

import torch

import torch_dist_ext_amd as tde

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "f64": torch.float64}
BYTES = {"bf16": 2, "f16": 2, "f32": 4, "f64": 8}
ALGOS = {"auto": tde.ALGO_AUTO, "staged": tde.ALGO_STAGED, "staged_owned": tde.ALGO_STAGED_OWNED}
STATIC_SCALE = 0.02  # a per-tensor scale of normed rows with gamma around 1: 448 * 0.02 is about nine standard deviations
MAX_BYTES = 2181249024  # the largest listed case's work


def _case(entry, nranks, tokens, hidden, dtype, quant, name=None, algo="auto", write_norm=False, eps=1e-6, sigma=1.0, outliers=False):
    c = dict(entry=entry, nranks=nranks, tokens=tokens, hidden=hidden, dtype=dtype, quant=quant, algo=algo,
             write_norm=write_norm, eps=eps, sigma=sigma, outliers=outliers)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest ordinary call: a few sequences of a small model, two ranks; launches and host time count
        _case("functional", 2, 16, 1024, "bf16", "none", name="small_16x1024"),
        # one decode step of a batch of 128 on eight ranks, T-typed output
        _case("functional", 8, 128, 4096, "bf16", "none", name="decode_128x4096", eps=1e-5, sigma=0.5),
        # a decode step and a mid-size batch of a model whose activations have outlier channels, int8 codes per token
        _case("functional", 4, 64, 5120, "f16", "int8_token", name="decode_64x5120_int8", outliers=True),
        _case("functional", 4, 512, 5120, "f16", "int8_token", name="batch_512x5120_int8", outliers=True),
        # prefill of 2048 tokens on eight ranks, fp8 codes per token: the headline configuration
        _case("functional", 8, 2048, 8192, "bf16", "fp8_token", name="prefill_2048x8192_fp8", eps=1e-5, sigma=0.5),
        # a long prefill with block scales into buffers that the serving loop keeps
        _case("in_place", 4, 8192, 7168, "bf16", "fp8_group", name="prefill_8192x7168_group"),
        # the largest call: 32768 tokens at once
        _case("functional", 4, 32768, 5120, "f16", "int8_token", name="sweep_32768x5120_int8", outliers=True),
        # many short rows that fill no whole number of wavefronts, fp32
        _case("functional", 8, 10024, 508, "f32", "none", name="rows_10024x508_f32"),
        # doubles (no quantized output exists for them)
        _case("functional", 4, 2048, 2048, "f64", "none", name="rows_2048x2048_f64"),
        # a ragged prefill on two ranks that wants both the codes of a calibrated static scale and the T-typed rows
        _case("partials", 2, 1257, 6144, "bf16", "fp8_static", name="ragged_1257x6144_static", write_norm=True),
        # the two-shot structure in one process: all rows summed into the stage, and one rank's share of it (the other
        # rows of the stage were delivered by the peers before the call)
        _case("partials", 8, 2048, 8192, "bf16", "fp8_token", name="staged_2048x8192_fp8", algo="staged", eps=1e-5, sigma=0.5),
        _case("partials", 8, 2048, 8192, "bf16", "fp8_token", name="owned_2048x8192_fp8", algo="staged_owned", eps=1e-5, sigma=0.5),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f16", "f32", "f64"])
        quant = "none" if dtype == "f64" else rng.choice(["none", "fp8_token", "fp8_group", "int8_token", "fp8_static"])
        entry = rng.choice(["functional", "functional", "in_place", "partials"])
        algo = rng.choice(["auto", "staged", "staged_owned"]) if entry == "partials" else "auto"
        nranks = rng.choice([2, 4, 8])
        # rows of 124 elements up to the longest the type allows (1024 vectors of 16 bytes), whole vectors; per-group
        # scales need whole groups of 128
        unit = 128 if quant == "fp8_group" else 16 // BYTES[dtype]
        hidden = max(unit, _log_uniform(rng, 124, 16384 // BYTES[dtype]) // unit * unit)
        tokens = _log_uniform(rng, 1, 32768)
        outliers = dtype == "f16" and quant == "int8_token"
        c = _case(entry, nranks, tokens, hidden, dtype, quant, algo=algo, write_norm=quant != "none" and rng.random() < 0.25,
                  eps=rng.choice([1e-5, 1e-6]), sigma=rng.choice([0.5, 1.0]), outliers=outliers)
        if work(c)["bytes"] <= MAX_BYTES:
            return c


class State:
    """One call's inputs and what a program keeps between calls: the workspace and its table, its own output buffers."""


def prepare(case, seed):
    dev, dtype = torch.device("cuda"), DTYPES[case["dtype"]]
    n, shape, mode = case["nranks"], (case["tokens"], case["hidden"]), tde.QUANT_MODES[case["quant"]]
    wide = torch.float64 if dtype == torch.float64 else torch.float32
    g = torch.Generator(device=dev).manual_seed(seed)
    s = State()
    s.entry, s.nranks, s.rank, s.eps, s.mode, s.write_norm = case["entry"], n, seed % n, case["eps"], mode, case["write_norm"]
    s.static_scale = STATIC_SCALE if mode == tde.QUANT_FP8_STATIC else 0.0
    s.algo, s.stage = ALGOS[case["algo"]], None
    # 0.1 % of the channels a hundred times larger, the same ones in every partial
    columns = torch.randperm(case["hidden"], generator=g, device=dev)[: max(1, case["hidden"] // 1000)] if case["outliers"] else None

    def partial():
        p = torch.randn(shape, generator=g, device=dev, dtype=wide).mul_(case["sigma"])
        if columns is not None:
            p[:, columns] *= 100.0
        return p.to(dtype)

    s.residual = torch.randn(shape, generator=g, device=dev, dtype=wide).to(dtype)
    s.gamma = (torch.rand(case["hidden"], generator=g, device=dev, dtype=wide) + 0.5).to(dtype)
    if s.entry == "partials":
        s.rank = 0
        s.partials = [partial() for _ in range(n)]
        if s.algo != tde.ALGO_AUTO:
            # the stage belongs to the caller; with owned rows the peers' rows of it are already there
            s.stage = (torch.randn(shape, generator=g, device=dev, dtype=wide) * (case["sigma"] * math.sqrt(n))).to(dtype)
        return s
    slot_bytes = -(-s.residual.numel() * s.residual.element_size() // 16) * 16
    s.comm = tde.CommWorkspace(s.rank, n, 256, slot_bytes)
    for r in range(n):
        p = partial()
        if r == s.rank:
            s.local = p
        else:
            s.comm.set_peer_partial(r, p)
    s.workspace = s.comm.get_workspace(s.local)
    if s.entry == "in_place":
        s.residual_out = torch.empty_like(s.residual)
        s.norm_out = torch.empty_like(s.residual) if mode == tde.QUANT_NONE or s.write_norm else None
        s.q_out = s.scale_out = None
        if mode != tde.QUANT_NONE:
            s.q_out = torch.empty(shape, device=dev, dtype=torch.int8 if mode == tde.QUANT_INT8_TOKEN else torch.float8_e4m3fn)
        if mode in (tde.QUANT_FP8_TOKEN, tde.QUANT_INT8_TOKEN):
            s.scale_out = torch.empty(shape[:1], device=dev, dtype=torch.float32)
        elif mode == tde.QUANT_FP8_GROUP:
            s.scale_out = torch.empty((shape[0], shape[1] // tde.QUANT_GROUP), device=dev, dtype=torch.float32)
    return s


def run(s):
    if s.entry == "functional":
        if s.mode == tde.QUANT_NONE:
            return tde.allreduce_rms(s.rank, s.nranks, s.local, s.residual, s.gamma, s.eps, s.workspace)
        return tde.allreduce_rms_quant(s.rank, s.nranks, s.local, s.residual, s.gamma, s.eps, s.workspace, s.mode, s.write_norm,
                                       s.static_scale)
    if s.entry == "in_place":
        if s.mode == tde.QUANT_NONE:
            tde.allreduce_rms_fusion_impl(s.rank, s.nranks, s.local, s.residual, s.gamma, s.residual_out, s.norm_out, s.eps,
                                          s.workspace)
        else:
            tde.allreduce_rms_quant_fusion_impl(s.rank, s.nranks, s.local, s.residual, s.gamma, s.residual_out, s.norm_out,
                                                s.q_out, s.scale_out, s.eps, s.workspace, s.mode, s.static_scale)
        return [s.residual_out, s.norm_out, s.q_out, s.scale_out]
    out = tde.reduce_rms(s.partials, s.residual, s.gamma, s.eps, s.mode, s.write_norm or s.mode == tde.QUANT_NONE, s.algo,
                         s.stage, s.static_scale)
    return [out, s.stage]


def work(case):
    """Each input read once, each output written once; the stage of the staged algorithms is an output (and, for the
    rows that the peers delivered, an input in the partials' place)."""
    n, t, h, e = case["nranks"], case["tokens"], case["hidden"], BYTES[case["dtype"]]
    row = h * e
    owned = -(-t // n) if case["algo"] == "staged_owned" else t  # rank 0's share of the rows
    read = owned * n * row + (t - owned) * row + t * row + row  # partials, delivered stage rows, residual, gamma
    written = t * row + (owned * row if case["algo"] != "auto" else 0)  # residual_out, summed stage rows
    if case["quant"] == "none" or case["write_norm"]:
        written += t * row
    if case["quant"] != "none":
        scales = {"fp8_token": t, "int8_token": t, "fp8_group": t * (h // 128), "fp8_static": 0}[case["quant"]]
        written += t * h + 4 * scales
    # per element: the additions, the square and its sum, two products of the norm, and for codes a quotient and a maximum
    flops = owned * h * n + t * h * (5 if case["quant"] == "none" else 7)
    return {"bytes": read + written, "flops": flops}


def tolerance(case):
    """Every output's bits are those of the torch-eager composition on the CPU (sums in rank order, the mean of squares in
    torch's own order, one rounding per step): compared with itself nothing differs."""
    return "exact"
