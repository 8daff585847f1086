"""Measured cases: the SVD-MLP work that users of this package have it do.

Every case is one call through the public entry points (``svdmlp.svd_mlp``,
``svd_mlp_block``, ``fused_gate_up``, ``fused_xuv``, ``compat.nki_mm``,
``stack.run_stack``).  A case is a dict of

    op         layer     y = xuv(gate_up(x)), one SVD-MLP layer
               block     x + layer(RMSNorm(x)), one MLP block of the model
               stack     `layers` blocks, each of its own ranks
               gate_up   the gate/up half alone
               xuv       the low-rank projection x . u . v alone (the down half)
    tokens     rows of x
    d, ff      hidden and intermediate size
    r_gate, r_up, r_down   ranks of the three low-rank factors (xuv: r_down)
    dtype      bf16, fp32, or fp8 (e4m3 factors with per-column scales, bf16 activations)
    layout     natural (U (d_in, r), V (r, d_out)), padded (natural, the V
               factors' rows 64 elements longer in memory), or linear
               (torch.nn.Linear weights as a checkpoint stores them)
    transposed (gate_up, xuv) h returned as (ff, tokens), x given as (ff, tokens)
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PACKAGE = Path(__file__).resolve().parent.parent / "neuronmlp-on-tpu_amd"
if str(_PACKAGE) not in sys.path:
    sys.path.insert(0, str(_PACKAGE))

import svdmlp  # noqa: E402
from svdmlp import compat, stack  # noqa: E402
from svdmlp.config import MODELS  # noqa: E402
from svdmlp.fp8 import quantize_per_channel  # noqa: E402
from svdmlp.ops import low_rank_dim, pad_rows  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32, "fp8": torch.bfloat16}
_EPS = 1e-5

# (d, ff) of the model shapes of svdmlp.config, and of the 8B layer's slice on
# each of eight ranks, the tiny test configuration and two mid-sized models
_SIZES = {name: (m.hidden_size, m.intermediate_size) for name, m in MODELS.items()}
_SIZES.update({"tiny": (1024, 3584), "slice": (4096, 1792), "small": (2048, 5632), "medium": (2560, 6912)})


def _case(op, tokens, d, ff, ranks, dtype="bf16", layout="natural", *, name=None, layers=1, transposed=False):
    c = {"op": op, "tokens": tokens, "d": d, "ff": ff, "r_gate": ranks[0], "r_up": ranks[1], "r_down": ranks[2],
         "dtype": dtype, "layout": layout, "layers": layers, "transposed": transposed}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one new token of one sequence through an 8B model's MLP block: the latency of every generated token
        _case("block", 1, 4096, 14336, (2816,) * 3, layout="padded", name="8b-block-decode-1"),
        # a small batch of sequences on a 3B model, factors as the operators' reference layout has them
        _case("layer", 8, 3072, 8192, (1792,) * 3, name="3b-layer-decode-8"),
        # a batch of 16 sequences on weights passed as the checkpoint's Linear tensors
        _case("layer", 16, 4096, 14336, (2816,) * 3, layout="linear", name="8b-linear-decode-16"),
        # a batch of 48 sequences: a server's ordinary decode step
        _case("block", 48, 4096, 14336, (2816,) * 3, layout="padded", name="8b-block-decode-48"),
        # decode of a 70B model, whose factors are kept in fp8
        _case("layer", 4, 8192, 28672, (5632,) * 3, dtype="fp8", name="70b-fp8-decode-4"),
        # the tiny fp32 configuration (numerics work, tests, CPU comparison)
        _case("layer", 128, 1024, 3584, (256,) * 3, dtype="fp32", name="tiny-fp32-128"),
        # the two halves as operators of their own: the transposed gate/up launcher on a short prompt ...
        _case("gate_up", 128, 4096, 14336, (2816,) * 3, transposed=True, name="8b-gate-up-t-128"),
        # ... and the low-rank projection on a decode batch
        _case("xuv", 32, 4096, 14336, (2816,) * 3, name="8b-xuv-32"),
        # a prompt of 512 tokens on a 3B model
        _case("layer", 512, 3072, 8192, (1792,) * 3, name="3b-layer-prefill-512"),
        # the headline: a 1024-token prompt through an 8B layer
        _case("layer", 1024, 4096, 14336, (2816,) * 3, layout="padded", name="8b-layer-prefill-1024"),
        # a long prompt of no round length through two blocks of a model compressed layer by layer
        _case("stack", 3001, 4096, 14336, (2304, 3072, 2560), layers=2, name="8b-stack-prefill-3001"),
        # a 70B prompt on fp8 factors, the largest call
        _case("layer", 2048, 8192, 28672, (5632,) * 3, dtype="fp8", name="70b-fp8-prefill-2048"),
    ]


def draw(rng):
    """One more case of the same ranges: operators, sizes, ranks, types and
    layouts drawn apart from each other, tokens over their logarithm."""
    dtype = rng.choice(("bf16",) * 6 + ("fp8",) * 2 + ("fp32",))
    op = rng.choice(("layer",) * 4 + ("block",) * 3 + ("stack", "gate_up", "xuv"))
    if dtype != "bf16" and op == "stack":
        op = "block"
    names = [n for n in _SIZES if dtype != "fp32" or n in ("tiny", "small", "slice")]
    d, ff = _SIZES[rng.choice(names)]
    # one rank at a compression ratio; now and then each factor its own, or
    # ranks off the 128 grid as a singular-value threshold picks them
    r = max(128, low_rank_dim(d, ff, rng.uniform(0.3, 0.9)))
    ranks = [r, r, r]
    pick = rng.random()
    if pick < 0.2 and op in ("layer", "block"):
        ranks = [max(128, r + 128 * rng.randint(-3, 3)) for _ in range(3)]
    elif pick < 0.35:
        ranks = [max(128, r - 8 * rng.randint(1, 15))] * 3
    layout = "natural"
    if dtype == "bf16" and op in ("layer", "block") and ranks[0] % 128 == 0:
        layout = rng.choice(("natural", "padded", "linear") if op == "layer" and ranks[0] == ranks[1]
                            else ("natural", "padded"))
    layers = rng.randint(2, 3) if op == "stack" else 1
    # no more work than the largest listed call
    most = {"bf16": 4096, "fp8": 2048, "fp32": 512}[dtype]
    budget = {"bf16": 1.6e12, "fp8": 2.0e12, "fp32": 5e10}[dtype]
    if layout == "linear" or ranks[0] % 128:
        budget /= 4
    per_token = _flops(_case(op, 1, d, ff, ranks, dtype, layers=layers))
    most = max(1, min(most, int(budget / per_token)))
    tokens = max(1, min(most, round(math.exp(rng.uniform(0.0, math.log(most + 0.5))))))
    return _case(op, tokens, d, ff, tuple(ranks), dtype, layout, layers=layers,
                 transposed=op in ("gate_up", "xuv") and rng.random() < 0.4)


def _draw_factor(g, rows, cols):
    return torch.randn(rows, cols, generator=g, device=g.device, dtype=torch.float32) / math.sqrt(rows)


def _activations(g, tokens, width, dtype):
    """Hidden states: unit normal per token with a spread of channel scales."""
    scale = torch.exp(0.5 * torch.randn(width, generator=g, device=g.device))
    return (torch.randn(tokens, width, generator=g, device=g.device) * scale).to(dtype)


def _layer_ranks(case):
    """(gate, up, down) ranks of each layer; a stack's layers rotate them."""
    r = (case["r_gate"], case["r_up"], case["r_down"])
    return [tuple(r[(i + j) % 3] for j in range(3)) for i in range(case["layers"])]


def _inputs(case, seed):
    """x, and per layer the factors (ug, vg, uu, vu, ud, vd) as stored
    (bf16 or fp32 tensors, or QuantizedFactor) and the RMSNorm gain."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    d, ff, dtype = case["d"], case["ff"], _DTYPES[case["dtype"]]

    def factor(rows, cols, is_v):
        w = _draw_factor(g, rows, cols)
        if case["dtype"] == "fp8":
            return quantize_per_channel(w)
        w = w.to(dtype)
        if case["layout"] == "padded" and is_v:
            return pad_rows(w)
        return w

    layers = []
    for rg, ru, rd in _layer_ranks(case):
        if case["op"] == "xuv":
            fs = (factor(ff, rd, False), factor(rd, d, True))
        else:
            fs = (factor(d, rg, False), factor(rg, ff, True), factor(d, ru, False), factor(ru, ff, True))
            if case["op"] != "gate_up":
                fs += (factor(ff, rd, False), factor(rd, d, True))
        gain = torch.rand(d, generator=g, device=g.device) * 0.2 + 0.9
        layers.append((gain, fs))
    if case["op"] == "xuv":  # the down half's input is h = silu(g) * u
        h = [torch.randn(case["tokens"], ff, generator=g, device=g.device) for _ in range(2)]
        x = (torch.nn.functional.silu(h[0]) * h[1]).to(dtype)
    else:
        x = _activations(g, case["tokens"], d, dtype)
    return x, layers


def prepare(case, seed):
    x, layers = _inputs(case, seed)
    state = {"case": case, "x": x}
    if case["op"] == "xuv" and case["transposed"]:
        state["x"] = x.t().contiguous()
    if case["op"] == "stack":
        # a model's layers, with the workspace and the two buffers that its loop keeps
        state["layers"] = [stack.StackLayer(gain, fs, r) for (gain, fs), r in zip(layers, _layer_ranks(case))]
        state["workspace"] = stack.stack_workspace(x, state["layers"])
        state["buffers"] = (torch.empty_like(x), torch.empty_like(x))
    else:
        state["gain"], state["factors"] = layers[0]
        if case["layout"] == "linear":
            state["factors"] = tuple(f.t().contiguous() for f in state["factors"])
    return state


def run(state):
    case, x = state["case"], state["x"]
    op = case["op"]
    if op == "stack":
        return stack.run_stack(x, state["layers"], eps=_EPS, workspace=state["workspace"], buffers=state["buffers"])
    f = state["factors"]
    if op == "gate_up":
        return svdmlp.fused_gate_up(x, *f, out_transposed=case["transposed"])
    if op == "xuv":
        return svdmlp.fused_xuv(x, *f, x_transposed=case["transposed"])
    if op == "block":
        return svdmlp.svd_mlp_block(x, state["gain"], *f, eps=_EPS)
    if case["layout"] == "linear":
        gate_v, gate_u, up_v, up_u, down_v, down_u = f
        return compat.nki_mm(x, up_v, up_u, gate_v, gate_u, down_v, down_u)
    return svdmlp.svd_mlp(x, *f)


def _flops(case):
    T, d, ff = case["tokens"], case["d"], case["ff"]
    total = 0
    for rg, ru, rd in _layer_ranks(case):
        if case["op"] != "xuv":
            total += 2 * T * (rg + ru) * (d + ff)
        if case["op"] != "gate_up":
            total += 2 * T * rd * (d + ff)
    return total


def work(case):
    T, d, ff = case["tokens"], case["d"], case["ff"]
    act = 4 if case["dtype"] == "fp32" else 2
    elem = {"bf16": 2, "fp32": 4, "fp8": 1}[case["dtype"]]
    values = columns = 0
    for rg, ru, rd in _layer_ranks(case):
        if case["op"] != "xuv":
            values += (rg + ru) * (d + ff)
            columns += rg + ru + 2 * ff
        if case["op"] != "gate_up":
            values += rd * (d + ff)
            columns += rd + d
    width_in = ff if case["op"] == "xuv" else d
    width_out = ff if case["op"] == "gate_up" else d
    factors = values * elem + (4 * columns if case["dtype"] == "fp8" else 0)
    gains = 4 * d * case["layers"] if case["op"] in ("block", "stack") else 0
    return {"bytes": factors + gains + T * (width_in + width_out) * act, "flops": _flops(case)}


def tolerance(case):
    # Four times the distance from 64 bits: bf16 rounds the rank
    # intermediates, h and the result once each (4e-3 to 5e-3 in the layer
    # and gate_up, 2.7e-3 in xuv); fp32 differs by the order of its sums.
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    return {"rel": 1e-2 if case["op"] == "xuv" else 2e-2}


def exact(case, seed):
    x, layers = _inputs(case, seed)

    def wide(f):
        if isinstance(f, svdmlp.QuantizedFactor):
            return f.data.double() * f.scale.double()
        return f.double()

    x = x.double()

    def gate_up(x, ug, vg, uu, vu):
        g = (x @ wide(ug)) @ wide(vg)
        return g * torch.sigmoid(g) * ((x @ wide(uu)) @ wide(vu))

    if case["op"] == "xuv":
        u, v = layers[0][1]
        return (x @ wide(u)) @ wide(v)
    if case["op"] == "gate_up":
        h = gate_up(x, *layers[0][1])
        return h.t().contiguous() if case["transposed"] else h
    for gain, fs in layers:
        inner = x
        if case["op"] != "layer":
            inner = x * torch.rsqrt((x * x).mean(dim=1, keepdim=True) + _EPS) * gain.double()
        y = (gate_up(inner, *fs[:4]) @ wide(fs[4])) @ wide(fs[5])
        x = y if case["op"] == "layer" else x + y
    return x
