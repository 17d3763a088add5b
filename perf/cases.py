"""The work a user of this framework has it do, as cases that can be timed: NVFP4 weights times activations through
``crow_nest_amd.engine.Engine``, from one small projection at one row to a prefill GEMM, and the encoder on the load path.

Weights are N(0, 0.02^2) encoded on the device by the framework's own encoder; activations are N(0, 1).  A decode case runs
several layers with weights of their own, because a decoder does: a single layer that is repeated would be read out of the
256 MB memory-side cache and not out of HBM.
"""
from __future__ import annotations

import math

import torch

from crow_nest_amd.engine import Engine, MlpW, MoeW, expert_table
from crow_nest_amd.kernels import KernelGeo
from crow_nest_amd.weights import ExpertSlabs, Fp4, dequant, load_fp4_quantized, quantize_nvfp4, repack_into, tiled_bytes

WEIGHT_STD = 0.02
BLOCK = 64          # NVFP4 container block: 64 values in 36 bytes
BLOCK_BYTES = 36


def listed():
    return [
        # the smallest call of a decode step: one small projection (a shared expert's) at one row - launch and host bound
        {"name": "proj_small", "kind": "proj", "t": 1, "rows": 512, "cols": 2048, "x": "f32", "layers": 1},
        # batch-1 dense projections of a 27B decoder, one tensor at a time
        {"name": "proj_decode", "kind": "proj", "t": 1, "rows": 17408, "cols": 5120, "x": "f32", "layers": 4},
        # three draft rows through a tensor whose rows and columns fill neither the last strip nor the last column group
        {"name": "proj_verify3_ragged", "kind": "proj", "t": 3, "rows": 6151, "cols": 3008, "x": "f32", "layers": 4},
        # batch-1 decode: gate/up + SiLU and down, bf16 activations
        {"name": "ffn_decode", "kind": "ffn", "t": 1, "hidden": 5120, "inter": 17408, "x": "bf16", "layers": 4},
        # the same at the widest speculative-verify width
        {"name": "ffn_verify4", "kind": "ffn", "t": 4, "hidden": 5120, "inter": 17408, "x": "bf16", "layers": 4},
        # the end of every decode step: logits over the vocabulary and the greedy token
        {"name": "head_greedy", "kind": "head", "rows": 151936, "cols": 5120},
        # batch-1 decode through routed layers: router projection, top-8 of 256 experts, combined
        {"name": "moe_decode", "kind": "moe", "t": 1, "experts": 256, "topk": 8, "hidden": 2048, "inter": 512, "layers": 8},
        # the same layers under a batch in which experts repeat
        {"name": "moe_batch64", "kind": "moe", "t": 64, "experts": 256, "topk": 8, "hidden": 2048, "inter": 512, "layers": 2},
        # a small batch (or a short prompt) through one projection
        {"name": "gemm_16", "kind": "gemm", "m": 16, "rows": 17408, "cols": 5120, "layers": 4},
        # prefill, one chunk of a prompt
        {"name": "gemm_512", "kind": "gemm", "m": 512, "rows": 17408, "cols": 5120, "layers": 1},
        # prefill of a long prompt through the down projection; a token count that fills no tile
        {"name": "gemm_1999_down", "kind": "gemm", "m": 1999, "rows": 5120, "cols": 17408, "layers": 1},
        # the load path: encode a tensor, lay it out for the kernels, decode it again (the converter's own check)
        {"name": "encode_decode", "kind": "encode", "rows": 17408, "cols": 5120},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _blocks(rng, lo: int, hi: int) -> int:
    """A number of columns: any whole number of container blocks."""
    return BLOCK * _log_int(rng, lo // BLOCK, hi // BLOCK)


_LARGEST_FLOPS = 2 * 1999 * 5120 * 17408  # the largest listed GEMM


def draw(rng):
    kind = rng.choice(["proj", "proj", "ffn", "ffn", "head", "moe", "moe", "gemm", "gemm", "gemm", "encode"])
    x = rng.choice(["f32", "bf16"])
    if kind == "proj":
        return {"kind": kind, "t": rng.randint(1, 4), "rows": _log_int(rng, 512, 20000), "cols": _blocks(rng, 1024, 17408), "x": x,
                "layers": rng.randint(1, 4)}
    if kind == "ffn":
        return {"kind": kind, "t": rng.randint(1, 4), "hidden": _blocks(rng, 1024, 8192), "inter": _blocks(rng, 2048, 17408), "x": x,
                "layers": rng.randint(1, 4)}
    if kind == "head":
        return {"kind": kind, "rows": _log_int(rng, 32000, 152000), "cols": _blocks(rng, 1024, 5120)}
    if kind == "moe":
        return {"kind": kind, "t": _log_int(rng, 1, 64), "experts": rng.choice([64, 128, 256]), "topk": rng.randint(4, 10),
                "hidden": _blocks(rng, 1024, 4096), "inter": _blocks(rng, 256, 768), "layers": rng.randint(1, 2)}
    if kind == "gemm":
        rows, cols = _log_int(rng, 1024, 17408), _blocks(rng, 1024, 17408)
        most = min(2048, _LARGEST_FLOPS // (2 * rows * cols))
        return {"kind": kind, "m": _log_int(rng, 5, most), "rows": rows, "cols": cols, "layers": 1}
    return {"kind": kind, "rows": _log_int(rng, 256, 17408), "cols": _blocks(rng, 1024, 5120)}


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, *shape, std: float = 1.0) -> torch.Tensor:
    return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, std, generator=gen)


def _tensor(gen, rows: int, cols: int) -> Fp4:
    blocks, gs = quantize_nvfp4(_normal(gen, rows, cols, std=WEIGHT_STD))
    return load_fp4_quantized(blocks, gs, rows, cols)


def _slabs(gen, experts: int, rows: int, cols: int) -> ExpertSlabs:
    blocks, gs = quantize_nvfp4(_normal(gen, experts, rows, cols, std=WEIGHT_STD))
    per, slab = rows * cols // BLOCK * BLOCK_BYTES, tiled_bytes(rows, cols)
    w = torch.empty(experts * slab, dtype=torch.uint8, device="cuda")
    for e in range(experts):
        repack_into(blocks[e * per:(e + 1) * per], rows, cols, w[e * slab:(e + 1) * slab])
    return ExpertSlabs(w, gs, experts, rows, cols, slab)


def _activations(gen, t: int, cols: int, kind: str) -> torch.Tensor:
    x = _normal(gen, t, cols)
    return x.to(torch.bfloat16) if kind == "bf16" else x


def prepare(case, seed):
    gen = _generator(seed)
    kind = case["kind"]
    state = {"kind": kind, "t": case.get("t", case.get("m", 1)), "layers": []}
    if kind == "encode":
        state["values"] = _normal(gen, case["rows"], case["cols"], std=WEIGHT_STD)
        return state
    if kind == "moe":
        e, h, i = case["experts"], case["hidden"], case["inter"]
        state["engine"] = Engine(KernelGeo(experts=e, topk=case["topk"], hidden=h, inter=i))
        for _ in range(case["layers"]):
            gate_up, down = _slabs(gen, e, 2 * i, h), _slabs(gen, e, h, i)
            router = _normal(gen, e, h, std=h ** -0.5)  # logits ~ N(0, 1)
            state["layers"].append((router, MoeW(gate_up, down, expert_table(gate_up, down)), _normal(gen, case["t"], h)))
        return state
    state["engine"] = Engine()
    if kind == "ffn":
        h, i = case["hidden"], case["inter"]
        for _ in range(case["layers"]):
            mlp = MlpW(_tensor(gen, i, h), _tensor(gen, i, h), _tensor(gen, h, i))
            state["layers"].append((mlp, _activations(gen, case["t"], h, case["x"])))
        return state
    x = {"proj": case.get("x"), "head": "f32", "gemm": "bf16"}[kind]
    for _ in range(case.get("layers", 1)):
        state["layers"].append((_tensor(gen, case["rows"], case["cols"]), _activations(gen, state["t"], case["cols"], x)))
    return state


def run(state):
    kind, t = state["kind"], state["t"]
    if kind == "encode":
        values = state["values"]
        rows, cols = values.shape
        blocks, gs = quantize_nvfp4(values)
        return blocks, gs, dequant(load_fp4_quantized(blocks, gs, rows, cols))
    eng = state["engine"]
    if kind == "proj":
        return [eng.dense_proj(w, t, x) for w, x in state["layers"]]
    if kind == "ffn":
        return [eng.dense_ffn_w(mlp, x, t) for mlp, x in state["layers"]]
    if kind == "head":
        return [eng.lm_head_row(w, x.view(-1)) for w, x in state["layers"]]
    if kind == "moe":
        return [eng.moe_layer(moe, x, eng.f32_proj(router, t, x)) for router, moe, x in state["layers"]]
    # a short prompt of up to four rows would go to the verify kernels; dense_proj takes every larger one to the GEMM
    return [eng.dense_proj(w, t, x) for w, x in state["layers"]]


def _decoded(gen, rows: int, cols: int) -> torch.Tensor:
    """f64 values of the container tensor that ``_tensor`` / ``_slabs`` would draw next: 36-byte blocks of four scale bytes
    (E4M3, 0x7F read as 448) and 32 bytes of two E2M1 codes each, the even value in the low nibble; times the global scale."""
    blocks, gs = quantize_nvfp4(_normal(gen, rows, cols, std=WEIGHT_STD))
    b = blocks.view(-1, BLOCK_BYTES)
    scales = (b[:, :4] & 0x7F).clamp(max=0x7E).contiguous().view(torch.float8_e4m3fn).to(torch.float64)
    codes = torch.stack((b[:, 4:] & 15, b[:, 4:] >> 4), dim=-1).view(-1, 4, 16)
    e2m1 = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64, device="cuda")
    return (e2m1[codes.long()] * scales.unsqueeze(-1) * gs.to(torch.float64)).view(rows, cols)


def _swiglu(gate_up: torch.Tensor, down: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    gate, up = (x @ gate_up.T).chunk(2, dim=-1)
    return (gate / (1.0 + torch.exp(-gate)) * up) @ down.T


def exact(case, seed):
    """The same inputs through plain torch in f64, from the container bytes on.  Expert ids, the greedy token and the
    encoder's bytes are whole numbers, its global scale is exact by definition: they have no such value."""
    gen = _generator(seed)
    kind = case["kind"]
    if kind == "encode":
        return None, None, _decoded(gen, case["rows"], case["cols"])
    out = []
    if kind == "moe":
        e, k, h, i, t = case["experts"], case["topk"], case["hidden"], case["inter"], case["t"]
        for _ in range(case["layers"]):
            gate_up, down = _decoded(gen, e * 2 * i, h).view(e, 2 * i, h), _decoded(gen, e * h, i).view(e, h, i)
            router = _normal(gen, e, h, std=h ** -0.5).to(torch.float64)
            x = _normal(gen, t, h).to(torch.float64)
            top, ids = (x @ router.T).topk(k, dim=-1)
            weights = torch.softmax(top, dim=-1)
            y = torch.zeros_like(x)
            for expert in ids.unique().tolist():
                rows, picks = (ids == expert).nonzero(as_tuple=True)
                y[rows] += weights[rows, picks].unsqueeze(-1) * _swiglu(gate_up[expert], down[expert], x[rows])
            out.append((None, weights, y))
        return out
    if kind == "ffn":
        h, i = case["hidden"], case["inter"]
        for _ in range(case["layers"]):
            gate, up, down = _decoded(gen, i, h), _decoded(gen, i, h), _decoded(gen, h, i)
            out.append(_swiglu(torch.cat((gate, up)), down, _activations(gen, case["t"], h, case["x"]).to(torch.float64)))
        return out
    x = {"proj": case.get("x"), "head": "f32", "gemm": "bf16"}[kind]
    t = case.get("t", case.get("m", 1))
    for _ in range(case.get("layers", 1)):
        w = _decoded(gen, case["rows"], case["cols"])
        y = _activations(gen, t, case["cols"], x).to(torch.float64) @ w.T
        out.append((y.view(-1), None) if kind == "head" else y)
    return out


def work(case):
    kind = case["kind"]
    layers = case.get("layers", 1)
    if kind == "encode":
        n = case["rows"] * case["cols"]
        # values in; container blocks, tiled tensor and decoded values out
        return {"bytes": 4 * n + 2 * n // BLOCK * BLOCK_BYTES + 4 * n, "flops": 0}
    if kind == "moe":
        t, e, k, h, i = case["t"], case["experts"], case["topk"], case["hidden"], case["inter"]
        touched = e * (1.0 - (1.0 - k / e) ** t)  # experts that at least one token picks, expected
        weights = touched * 3 * h * i / BLOCK * BLOCK_BYTES
        return {"bytes": layers * (weights + 4 * e * h + 2 * 4 * t * h), "flops": layers * 2 * t * (e * h + k * 3 * h * i)}
    if kind == "ffn":
        t, h, i = case["t"], case["hidden"], case["inter"]
        x_bytes = 2 if case["x"] == "bf16" else 4
        return {"bytes": layers * (3 * h * i // BLOCK * BLOCK_BYTES + t * h * (x_bytes + 4)), "flops": layers * 2 * t * 3 * h * i}
    t = case.get("t", case.get("m", 1))
    rows, cols = case["rows"], case["cols"]
    x_bytes = 2 if kind == "gemm" or case.get("x") == "bf16" else 4
    return {"bytes": layers * (rows * cols // BLOCK * BLOCK_BYTES + t * (cols * x_bytes + rows * 4)), "flops": layers * 2 * t * rows * cols}


def tolerance(case):
    """Sums of K products in f32, in whatever order: against the same products in f64 the listed cases show a relative error
    (2-norm) of 1e-7 (GEMV, FFN, GEMM at 16 rows) to 4.6e-7 (GEMM, K = 17408) and a largest one of 3e-7 to 4.7e-6; four times
    that is stated.  The encoder's bytes and the decoded values are exact."""
    if case["kind"] == "encode":
        return "exact"
    return {"rel": 2e-6, "max": 2e-5}
