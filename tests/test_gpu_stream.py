"""The streaming stages of decode shapes (csrc/stream.hpp): Linear-layout and
fp8 factors, dimensions off the decode layer's tiles, and the gate/up and
x.u.v entry points, at the edges of their tiles.

Tolerance: bf16 results round the rank intermediate, h and y once each, a
relative error of at most 2^-9 per value and rounding (rms 1.1e-3); through
the layer's products and SiLU(g) * u the three add up to 3e-3 to 6e-3 of the
result's norm, so 1e-2.  fp8 factors are widened exactly and are compared
with the same math on the dequantised factors.
"""

import numpy as np
import pytest
import torch

import oracle as O
from svdmlp import _lib, fp8, inputs, ops

pytestmark = pytest.mark.gpu

TOL = 1e-2


def _np(t):
    return t.float().cpu().numpy()


def _rel(got, want):
    return float(np.linalg.norm(got - want) / np.linalg.norm(want))


def _layer(shape, T, seed, kind, dev):
    """(x, factors) as the operators take them and as float32 arrays."""
    x, f = inputs.make_layer(shape, T=T, seed=seed)
    xb = inputs.as_float32(x, torch.bfloat16)
    xt = inputs.to_torch(xb, torch.bfloat16, dev)
    if kind == "fp8":
        q = [fp8.quantize_per_channel(torch.from_numpy(a)) for a in f]
        wide = [O.e4m3_decode(a.data.view(torch.uint8).numpy()) * a.scale.numpy() for a in q]
        return xb, wide, xt, [ops.QuantizedFactor(a.data.to(dev), a.scale.to(dev)) for a in q]
    wide = [inputs.as_float32(a, torch.bfloat16) for a in f]
    ft = [inputs.to_torch(a, torch.bfloat16, dev) for a in wide]
    if kind == "linear":
        ft = [a.t().contiguous().t() for a in ft]
    return xb, wide, xt, ft


# 16-row token tiles full, one over and short of full; ranks and widths off the
# 128-column (fp8: 256) tiles, off the 64-k blocks and 32-k steps and down to
# one 8-wide piece; more K splits than one batch of slices (d = 4160: 16)
@pytest.mark.parametrize("T", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("kind", ["natural", "linear", "fp8"])
@pytest.mark.parametrize("shape", [inputs.LayerShape(136, 200, 72, 40), inputs.LayerShape(4160, 528, 136, 264),
                                   inputs.LayerShape(264, 2064, 400, 272)])
def test_stream_entry_points(gpu, shape, kind, T):
    xb, wide, xt, ft = _layer(shape, T, 300 + T, kind, gpu)
    h = ops.fused_gate_up(xt, *ft[:4])
    assert _rel(_np(h), O.fused_gate_up_ref(xb, *wide[:4], dtype="bfloat16")) < TOL
    y = ops.fused_xuv(h, *ft[4:])
    assert _rel(_np(y), O.fused_xuv_ref(_np(h), *wide[4:], dtype="bfloat16")) < TOL
    out = ops.svd_mlp(xt, *ft)
    assert _rel(_np(out), O.svd_mlp_ref(xb, *wide, dtype="bfloat16")) < TOL
    # split-K slices are summed in split order whichever unit is last: the same bits on replay
    for _ in range(3):
        assert torch.equal(ops.fused_gate_up(xt, *ft[:4]).view(torch.int16), h.view(torch.int16))
        assert torch.equal(ops.svd_mlp(xt, *ft).view(torch.int16), out.view(torch.int16))
    if T % 8 == 0 or kind != "fp8":  # transposed operands (fp8: T % 8 == 0 only): the natural result's bits
        hT = ops.fused_gate_up(xt, *ft[:4], out_transposed=True)
        assert torch.equal(hT.view(torch.int16), h.t().contiguous().view(torch.int16))
        yT = ops.fused_xuv(h.t().contiguous(), *ft[4:], x_transposed=True)
        assert torch.equal(yT.view(torch.int16), y.view(torch.int16))


# Linear factors at one and two tokens (csrc/gemv_linear.hip): K of one 8-wide
# piece, short of and past one 512-k step, one batch of steps and two batches;
# the block's residual; the same bits on replay and with a single token's row
# in a call of two.
@pytest.mark.parametrize("shape", [inputs.LayerShape(8, 16, 8), inputs.LayerShape(520, 1032, 504, 2056),
                                   inputs.LayerShape(2048, 4104, 1160, 1032), inputs.LayerShape(4096, 8200, 72)])
@pytest.mark.parametrize("T", [1, 2])
def test_linear_gemv(gpu, shape, T):
    xb, wide, xt, ft = _layer(shape, T, 60 + T, "linear", gpu)
    h = ops.fused_gate_up(xt, *ft[:4])
    assert _rel(_np(h), O.fused_gate_up_ref(xb, *wide[:4], dtype="bfloat16")) < TOL
    y = ops.fused_xuv(h, *ft[4:])
    assert _rel(_np(y), O.fused_xuv_ref(_np(h), *wide[4:], dtype="bfloat16")) < TOL
    out = ops.svd_mlp(xt, *ft)
    assert _rel(_np(out), O.svd_mlp_ref(xb, *wide, dtype="bfloat16")) < TOL
    assert torch.equal(ops.svd_mlp(xt, *ft).view(torch.int16), out.view(torch.int16))
    assert torch.equal(ops.svd_mlp(xt[:1].contiguous(), *ft).view(torch.int16), out[:1].view(torch.int16))
    gain = torch.rand(shape.d, device=gpu) + 0.5
    xn = (xt.float() * torch.rsqrt(xt.float().pow(2).mean(1, keepdim=True) + 1e-5) * gain).bfloat16()
    want = (xt.float() + ops.svd_mlp(xn, *ft).float()).bfloat16()
    assert _rel(_np(ops.svd_mlp_block(xt, gain, *ft)), _np(want)) < TOL


# 65-128 tokens: a second group of token rows with units, slices and tile
# counters of its own, from one row to full; K splits (d = 4160) and none,
# dimensions that the large tiles take (512, 1024) and not, the transposed
# result, the block's residual.
@pytest.mark.parametrize("T", [65, 72, 113, 128])
@pytest.mark.parametrize("kind", ["natural", "linear", "fp8"])
@pytest.mark.parametrize("shape", [inputs.LayerShape(136, 200, 72, 40), inputs.LayerShape(4160, 528, 136, 264),
                                   inputs.LayerShape(264, 2064, 400, 272), inputs.LayerShape(512, 1024, 160)])
def test_stream_two_row_groups(gpu, shape, kind, T):
    xb, wide, xt, ft = _layer(shape, T, 900 + T, kind, gpu)
    h = ops.fused_gate_up(xt, *ft[:4])
    assert _rel(_np(h), O.fused_gate_up_ref(xb, *wide[:4], dtype="bfloat16")) < TOL
    y = ops.fused_xuv(h, *ft[4:])
    assert _rel(_np(y), O.fused_xuv_ref(_np(h), *wide[4:], dtype="bfloat16")) < TOL
    ops.clear_workspace_cache()
    out = ops.svd_mlp(xt, *ft)
    assert _rel(_np(out), O.svd_mlp_ref(xb, *wide, dtype="bfloat16")) < TOL
    for _ in range(3):
        assert torch.equal(ops.svd_mlp(xt, *ft).view(torch.int16), out.view(torch.int16))
    (ws,) = ops._WS_CACHE.values()
    assert not any(ws[2560:4096].view(torch.int32).cpu().tolist())
    if T % 8 == 0 or kind != "fp8":
        hT = ops.fused_gate_up(xt, *ft[:4], out_transposed=True)
        assert torch.equal(hT.view(torch.int16), h.t().contiguous().view(torch.int16))
        yT = ops.fused_xuv(h.t().contiguous(), *ft[4:], x_transposed=True)
        assert torch.equal(yT.view(torch.int16), y.view(torch.int16))
    gain = torch.rand(shape.d, device=gpu) + 0.5
    xn = (xt.float() * torch.rsqrt(xt.float().pow(2).mean(1, keepdim=True) + 1e-5) * gain).bfloat16()
    want = (xt.float() + ops.svd_mlp(xn, *ft).float()).bfloat16()
    assert _rel(_np(ops.svd_mlp_block(xt, gain, *ft)), _np(want)) < TOL


def test_stream_two_row_groups_leave_padded_factors(gpu):
    """Factors with padded rows stay on the large tiles, which know the pitch."""
    xb, wide, xt, ft = _layer(inputs.LayerShape(512, 1024, 160), 100, 15, "natural", gpu)
    padded = [ops.pad_rows(a) if i % 2 else a for i, a in enumerate(ft)]
    assert padded[1].stride(0) > padded[1].shape[1]
    assert _rel(_np(ops.svd_mlp(xt, *padded)), O.svd_mlp_ref(xb, *wide, dtype="bfloat16")) < TOL


@pytest.mark.parametrize("kind", ["linear", "fp8"])
def test_stream_block(gpu, kind):
    """The MLP block: RMSNorm ahead, the residual added by the last stage."""
    shape = inputs.LayerShape(1024, 2048, 512, 384)
    xb, wide, xt, ft = _layer(shape, 24, 11, kind, gpu)
    gain = torch.rand(shape.d, device=gpu) + 0.5
    y = ops.svd_mlp_block(xt, gain, *ft)
    mlp = ops.svd_mlp((xt.float() * torch.rsqrt(xt.float().pow(2).mean(1, keepdim=True) + 1e-5) * gain).bfloat16(), *ft)
    # bf16(x + bf16(mlp)); the RMSNorm's own rounding may differ by one bf16 step
    assert _rel(_np(y), _np((xt.float() + mlp.float()).bfloat16())) < TOL


def test_stream_small_workspace(gpu):
    """A workspace without the larger slice area at its end (fewer K splits)."""
    shape = inputs.LayerShape(1024, 2048, 512)
    xb, wide, xt, ft = _layer(shape, 16, 12, "linear", gpu)
    ws = ops.svd_mlp_workspace(xt, r=shape.r, ff=shape.ff)
    extra = 16 * 1024 * 128 * 4
    short = torch.zeros(ws.numel() - extra, dtype=torch.uint8, device=gpu)
    want = O.svd_mlp_ref(xb, *wide, dtype="bfloat16")
    for w in (ws, short):
        assert _rel(_np(ops.svd_mlp(xt, *ft, workspace=w)), want) < TOL


@pytest.mark.parametrize("kind", ["linear", "fp8"])
def test_stream_workspace_of_more_tokens(gpu, kind):
    """The bits do not depend on which larger token count the workspace is for."""
    shape = inputs.LayerShape(2048, 8192, 1792)
    xb, wide, xt, ft = _layer(shape, 30, 17, kind, gpu)
    code = _lib.SVDMLP_FP8_E4M3 if kind == "fp8" else _lib.SVDMLP_BF16
    want = ops.svd_mlp(xt, *ft, workspace=ops.svd_mlp_workspace(xt, r=shape.r, ff=shape.ff, w_code=code))
    for T in (33, 64, 65):
        more = torch.empty(T, shape.d, dtype=xt.dtype, device=gpu)
        ws = ops.svd_mlp_workspace(more, r=shape.r, ff=shape.ff, w_code=code)
        assert torch.equal(ops.svd_mlp(xt, *ft, workspace=ws).view(torch.int16), want.view(torch.int16)), T


def test_stream_after_a_timeout(gpu):
    """A workspace whose timeout flag is set gives NaN until it is reset (the
    tile counters may hold anything then)."""
    shape = inputs.LayerShape(1024, 2048, 512)
    xb, wide, xt, ft = _layer(shape, 8, 13, "linear", gpu)
    ws = ops.svd_mlp_workspace(xt, r=shape.r, ff=shape.ff)
    ws[2304:2312].view(torch.int64).fill_(1)
    assert torch.isnan(ops.svd_mlp(xt, *ft, workspace=ws)).all()
    assert ops.workspace_status(ws, reset=True) is True
    assert _rel(_np(ops.svd_mlp(xt, *ft, workspace=ws)), O.svd_mlp_ref(xb, *wide, dtype="bfloat16")) < TOL


def _flag_timeout(ws):
    """The sync area as a timed-out persistent call may leave it."""
    ws[2560:4096] = torch.arange(1536, device=ws.device).mul(37).remainder(251).to(torch.uint8)
    ws[2304:2312].view(torch.int64).fill_(1)


# The halves and fp32 calls have no waits: on a workspace whose timeout flag is
# set, and whose tile counters hold anything, they compute as ever.  Stages
# with K splits (d = 4160, fp8 in 256-column tiles among them) and without,
# two row groups, the transposed result; fp32 from one token to several tiles.
@pytest.mark.parametrize("T", [1, 16, 40, 72, 100])
@pytest.mark.parametrize("kind", ["natural", "linear", "fp8"])
def test_stream_halves_after_a_timeout(gpu, kind, T):
    xb, wide, xt, ft = _layer(inputs.LayerShape(4160, 528, 136, 264), T, 30 + T, kind, gpu)
    ops.clear_workspace_cache()
    try:
        h = ops.fused_gate_up(xt, *ft[:4])
        ops.fused_xuv(h, *ft[4:])
        for ws in ops._WS_CACHE.values():
            _flag_timeout(ws)
        h = ops.fused_gate_up(xt, *ft[:4])
        assert _rel(_np(h), O.fused_gate_up_ref(xb, *wide[:4], dtype="bfloat16")) < TOL
        y = ops.fused_xuv(h, *ft[4:])
        assert _rel(_np(y), O.fused_xuv_ref(_np(h), *wide[4:], dtype="bfloat16")) < TOL
        if T % 8 == 0:
            assert torch.equal(ops.fused_gate_up(xt, *ft[:4], out_transposed=True).t(), h)
        assert ops.workspace_status() is True
    finally:
        ops.clear_workspace_cache()


@pytest.mark.parametrize("T", [1, 17, 128, 300])
@pytest.mark.parametrize("kind", ["natural", "linear"])
def test_f32_after_a_timeout(gpu, kind, T):
    shape = inputs.LayerShape(1024, 3584, 256)
    x, f = inputs.make_layer(shape, T=T, seed=600 + T)
    xt, ft = torch.from_numpy(x).to(gpu), [torch.from_numpy(a).to(gpu) for a in f]
    if kind == "linear":
        ft = [a.t().contiguous().t() for a in ft]
    ws = ops.svd_mlp_workspace(xt, r=shape.r, ff=shape.ff)
    _flag_timeout(ws)
    w = [a.double() for a in ft]
    g = (xt.double() @ w[0]) @ w[1]
    want = ((g * torch.sigmoid(g) * ((xt.double() @ w[2]) @ w[3])) @ w[4]) @ w[5]
    assert float((ops.svd_mlp(xt, *ft, workspace=ws).double() - want).norm() / want.norm()) < 1e-5


def test_fp8_transposed_odd_tokens_stay_refused(gpu):
    _, _, xt, ft = _layer(inputs.LayerShape(264, 528, 136), 9, 14, "fp8", gpu)
    for call in (lambda: ops.fused_gate_up(xt, *ft[:4], out_transposed=True),
                 lambda: ops.fused_xuv(torch.zeros(528, 9, dtype=torch.bfloat16, device=gpu), *ft[4:], x_transposed=True)):
        with pytest.raises(ValueError, match="multiples of 8"):
            call()


def test_stream_two_streams(gpu):
    """Two streams at once, a workspace each: no unit waits for another."""
    shape = inputs.LayerShape(2048, 4096, 512)
    sets = [_layer(shape, T, 20 + T, kind, gpu) for T, kind in ((16, "fp8"), (40, "linear"))]
    ws = [ops.svd_mlp_workspace(s[2], r=shape.r, ff=shape.ff, w_code=_lib.SVDMLP_BF16) for s in sets]
    want = [ops.svd_mlp(s[2], *s[3], workspace=w).clone() for s, w in zip(sets, ws)]
    streams = [torch.cuda.Stream() for _ in sets]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(20):
        for i, st in enumerate(streams):
            with torch.cuda.stream(st):
                got[i].append(ops.svd_mlp(sets[i][2], *sets[i][3], workspace=ws[i]))
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(g.view(torch.int16), want[i].view(torch.int16)) for g in got[i])


# fp32 stages (csrc/stream_f32.hpp).  Tolerance: a product over K terms summed
# in fp32 is off by at most about sqrt(K) 2^-24 of its norm, 7e-6 at K = 14336
# and less at these sizes; three products in a row and SiLU's reciprocal
# (1 ulp) stay below 1e-5.
@pytest.mark.parametrize("T", [1, 16, 17, 64, 65, 130, 300])
@pytest.mark.parametrize("kind", ["natural", "linear"])
@pytest.mark.parametrize("shape", [inputs.LayerShape(136, 200, 72, 40), inputs.LayerShape(1024, 3584, 256),
                                   inputs.LayerShape(264, 1040, 392, 8)])
def test_f32_stages(gpu, shape, kind, T):
    x, f = inputs.make_layer(shape, T=T, seed=500 + T)
    xt = torch.from_numpy(x).to(gpu)
    ft = [torch.from_numpy(a).to(gpu) for a in f]
    if kind == "linear":
        ft = [a.t().contiguous().t() for a in ft]
    w = [a.double() for a in ft]
    g = (xt.double() @ w[0]) @ w[1]
    h64 = g * torch.sigmoid(g) * ((xt.double() @ w[2]) @ w[3])
    rel = lambda a, b: float((a.double() - b).norm() / b.norm())  # noqa: E731
    h = ops.fused_gate_up(xt, *ft[:4])
    assert rel(h, h64) < 1e-5
    y = ops.fused_xuv(h, *ft[4:])
    assert rel(y, (h.double() @ w[4]) @ w[5]) < 1e-5
    out = ops.svd_mlp(xt, *ft)
    assert rel(out, (h64 @ w[4]) @ w[5]) < 1e-5
    assert torch.equal(ops.svd_mlp(xt, *ft), out)
    # transposed operands: the same sums
    assert torch.equal(ops.fused_gate_up(xt, *ft[:4], out_transposed=True), h.t())
    assert torch.equal(ops.fused_xuv(h.t().contiguous(), *ft[4:], x_transposed=True), y)
    gain = torch.rand(shape.d, device=gpu) + 0.5
    xn = xt.double() * torch.rsqrt(xt.double().pow(2).mean(1, keepdim=True) + 1e-5) * gain.double()
    g = (xn @ w[0]) @ w[1]
    want = xt.double() + ((g * torch.sigmoid(g) * ((xn @ w[2]) @ w[3])) @ w[4]) @ w[5]
    assert rel(ops.svd_mlp_block(xt, gain, *ft), want) < 1e-5


# SiLU over the range of its exponential.  U and V are identities, so the gate
# and the up value are x itself.  For x < 0 exp(-x) carries the rounding of its
# argument, |x| 2^-24 relative and as much again for the log2(e) it is
# multiplied with, and 1 + exp(-x), the reciprocal and the two products a unit
# in the last place each; from about -87.3 on the reciprocal would be
# subnormal and the result is zero, |x| 2^-126 off at most.
@pytest.mark.parametrize("T", [3, 200])
def test_silu_over_the_range_of_its_exponential(gpu, T):
    d = 256
    x = torch.linspace(-110, 110, T * d, device=gpu, dtype=torch.float64).float().reshape(T, d)
    eye = torch.eye(d, device=gpu)
    got = ops.fused_gate_up(x, eye, eye, eye, eye).double()
    x = x.double()
    want = x * torch.sigmoid(x) * x
    bound = want.abs() * (2 * x.abs() + 16) * 2.0**-24 + x * x * 2.0**-126
    assert ((got - want).abs() <= bound).all()


# The persistent decode layer's phase 2 in K splits (layers narrower than the
# grid): 2 (3B-like ratio) and 9 (ff = 1792, rank 2304) ways, distinct gate and
# up ranks whose splits end apart, the last-arrival (up to 16 tokens) and the
# shared form, and eight token tiles (phase 3 on its K splits' h flags).
@pytest.mark.parametrize("T", [4, 16, 17, 48, 100, 128])
@pytest.mark.parametrize("ranks", [(512, 512, 256), (2304, 1152, 384)])
@pytest.mark.parametrize("d,ff", [(1024, 8192), (512, 1792)])
def test_decode_layer_phase2_splits(gpu, d, ff, ranks, T):
    rng = np.random.default_rng(T + ff)
    rg, ru, rd = ranks
    mats = [inputs.random_matrix(rng, *s) for s in ((d, rg), (rg, ff), (d, ru), (ru, ff), (ff, rd), (rd, d))]
    wide = [inputs.as_float32(a, torch.bfloat16) for a in mats]
    xb = inputs.as_float32(rng.normal(size=(T, d)).astype(np.float32), torch.bfloat16)
    xt, ft = inputs.to_torch(xb, torch.bfloat16, gpu), [inputs.to_torch(a, torch.bfloat16, gpu) for a in wide]
    want = O.svd_mlp_ref(xb, *wide, dtype="bfloat16")
    ops.clear_workspace_cache()
    out = ops.svd_mlp(xt, *ft)
    assert _rel(_np(out), want) < TOL
    for _ in range(3):
        assert torch.equal(ops.svd_mlp(xt, *ft).view(torch.int16), out.view(torch.int16))
    (ws,) = ops._WS_CACHE.values()
    assert not any(ws[2560:4096].view(torch.int32).cpu().tolist()) and not ops.workspace_status()


# Large-tile path with ranks off the 32-k stages (XU held in whole 64-column
# blocks, the last one the last 64 ranks with zeros for those it repeats): one
# rank piece past a block (72), one short of it (504 = 7 * 64 + 56), in and off
# the 16 columns of an fp8 piece, equal and different down ranks; token counts
# of every plan (split passes, K-group tiles, one launch of both passes).
@pytest.mark.parametrize("T", [65, 128, 200, 300, 520, 1030])
@pytest.mark.parametrize("kind", ["natural", "linear", "fp8"])
@pytest.mark.parametrize("shape", [inputs.LayerShape(1024, 2048, 336, 504), inputs.LayerShape(256, 1792, 72, 1160),
                                   inputs.LayerShape(512, 4096, 496, 80)])
def test_ranks_off_the_stages(gpu, shape, kind, T):
    xb, wide, xt, ft = _layer(shape, T, 700 + T, kind, gpu)
    h = ops.fused_gate_up(xt, *ft[:4])
    assert _rel(_np(h), O.fused_gate_up_ref(xb, *wide[:4], dtype="bfloat16")) < TOL
    y = ops.fused_xuv(h, *ft[4:])
    assert _rel(_np(y), O.fused_xuv_ref(_np(h), *wide[4:], dtype="bfloat16")) < TOL
    out = ops.svd_mlp(xt, *ft)
    assert _rel(_np(out), O.svd_mlp_ref(xb, *wide, dtype="bfloat16")) < TOL
    if kind != "fp8" or shape.rd % 16 == 0:  # (the general kernel, which sums K splits by float atomics, has the others)
        assert torch.equal(ops.svd_mlp(xt, *ft).view(torch.int16), out.view(torch.int16))
    if kind == "natural":
        gain = torch.rand(shape.d, device=gpu) + 0.5
        blk = ops.svd_mlp_block(xt, gain, *ft)
        xn = (xt.float() * torch.rsqrt(xt.float().pow(2).mean(1, keepdim=True) + 1e-5) * gain).bfloat16()
        assert _rel(_np(blk), _np((xt.float() + ops.svd_mlp(xn, *ft).float()).bfloat16())) < TOL


# e4m3 h (SVDMLP_FP8_ACT) is for ranks in whole 32-k stages: with the gate/up
# or the down rank off them the layer runs as without the flag, to its bits.
@pytest.mark.parametrize("T", [65, 128, 300])
@pytest.mark.parametrize("shape", [inputs.LayerShape(512, 1024, 336, 256), inputs.LayerShape(512, 1024, 256, 336)])
def test_ranks_off_the_stages_keep_bf16_h(gpu, shape, T):
    xb, wide, xt, ft = _layer(shape, T, 40 + T, "fp8", gpu)
    got = ops.svd_mlp(xt, *ft, fp8_activations=True)
    assert _rel(_np(got), O.svd_mlp_ref(xb, *wide, dtype="bfloat16")) < TOL
    if T > 128:  # (below, the flag keeps the large tiles where the streaming stages are the default)
        assert torch.equal(got.view(torch.int16), ops.svd_mlp(xt, *ft).view(torch.int16))


# An infinite weight among the rows that the last 64-rank block repeats gives
# infinities by the sign of its rank value, not NaN (infinity times zero).
@pytest.mark.parametrize("T", [65, 300, 1030])
@pytest.mark.parametrize("kind", ["natural", "linear"])
@pytest.mark.parametrize("r", [72, 336, 504])
def test_ranks_off_the_stages_infinite_weight(gpu, r, kind, T):
    d, ff = 512, 1024
    rng = np.random.default_rng(T + r)
    u = torch.from_numpy(np.eye(d, dtype=np.float32)[:, :r].copy()).to(gpu, torch.bfloat16)
    v = torch.from_numpy(inputs.random_matrix(rng, r, ff)).to(gpu, torch.bfloat16)
    v[r - 64, 5] = float("inf")
    v[(r - 1) // 64 * 64 - 1, 700] = float("-inf")
    x = torch.from_numpy(rng.choice([-1.5, 0.75, 2.0], size=(T, d)).astype(np.float32)).to(gpu, torch.bfloat16)
    want = x.float().cpu()[:, :r] @ v.float().cpu()
    if kind == "linear":
        u, v = u.t().contiguous().t(), v.t().contiguous().t()
    got = ops.fused_xuv(x, u, v).float().cpu()
    assert torch.equal(torch.isposinf(got), torch.isposinf(want)) and torch.equal(torch.isneginf(got), torch.isneginf(want))
    assert torch.isfinite(got).sum() == T * (ff - 2)


# An infinite activation: the rank columns that the last 64-rank block repeats
# hold zeros for XU's gap, not the NaN of infinity times a zero weight.  U and
# V of one sign keep the results infinite.  Split and unsplit X.U products of
# every tile width, natural and Linear factors.
@pytest.mark.parametrize("T", [65, 130, 300, 1030])
@pytest.mark.parametrize("kind", ["natural", "linear", "fp8"])
@pytest.mark.parametrize("r", [80, 336, 504, 1104])
def test_ranks_off_the_stages_infinite_activation(gpu, r, kind, T):
    d, ff = 512, 1024
    rng = np.random.default_rng(T + r)
    f = [torch.from_numpy(np.abs(inputs.random_matrix(rng, *s)) + 0.01) for s in ((d, r), (r, ff), (d, r), (r, ff), (ff, r), (r, d))]
    x = torch.from_numpy(np.abs(rng.normal(size=(T, d))).astype(np.float32))
    rows = [3, T // 2, T - 1]
    for i, m in enumerate(rows):
        x[m, 7 * i] = float("inf")
    x = x.to(gpu, torch.bfloat16)
    if kind == "fp8":
        f = [fp8.quantize_per_channel(a.to(gpu)) for a in f]
    else:
        f = [a.to(gpu, torch.bfloat16) for a in f]
        if kind == "linear":
            f = [a.t().contiguous().t() for a in f]
    for got in (ops.fused_xuv(x, f[0], f[1]), ops.fused_gate_up(x, *f[:4]), ops.svd_mlp(x, *f)):
        got = got.float().cpu()
        inf = torch.isposinf(got)
        assert inf[rows].all() and torch.isfinite(got).sum() == got.numel() - inf[rows].numel()


# 129-256 tokens where the 128 x 128 K-group tiles fill at most half the CUs:
# the branches as batch entries in 1, 2 and 4 K splits (the last one ragged at
# rank 1088 and 2112), ragged last row tiles, the transposed result, a rank at
# the line (512) and one below it (448: both branches in a block).
@pytest.mark.parametrize("T", [129, 200, 256])
@pytest.mark.parametrize("ff,r", [(1792, 1088), (1792, 2112), (8192, 512), (8192, 448), (128, 2048)])
def test_gate_up_paired_kgroup_tiles(gpu, ff, r, T):
    xb, wide, xt, ft = _layer(inputs.LayerShape(512, ff, r, 128), T, T + r, "natural", gpu)
    h = ops.fused_gate_up(xt, *ft[:4])
    assert _rel(_np(h), O.fused_gate_up_ref(xb, *wide[:4], dtype="bfloat16")) < TOL
    assert torch.equal(ops.fused_gate_up(xt, *ft[:4]).view(torch.int16), h.view(torch.int16))
    if T % 8 == 0:
        assert torch.equal(ops.fused_gate_up(xt, *ft[:4], out_transposed=True).t(), h)
    assert _rel(_np(ops.svd_mlp(xt, *ft)), O.svd_mlp_ref(xb, *wide, dtype="bfloat16")) < TOL


# The gate values stay in 32 bits up to SiLU for ranks off the stages and for
# transposed results at token counts off 8.  U holds one-hot columns, so XU is
# exact and h is one rounding to bf16 from 64 bits: its error over the one of a
# correctly rounded h is the fp32 sums' (1e-5 of it), where a gate value
# rounded to bf16 on the way would bring sqrt(2) times the error.  fn 4, 7 and
# 8 tiles (ff = 2048 / 1792), split and unsplit, natural, Linear and fp8.
@pytest.mark.parametrize("T", [65, 131, 300, 500, 515, 1030])
@pytest.mark.parametrize("kind,ff,r", [(k, ff, r) for k in ("natural", "linear", "fp8")
                                       for ff, r in ((2048, 336), (1792, 528), (1800, 80), (2048, 256))
                                       if k != "fp8" or r % 32])  # fp8: no transposed result at such counts
def test_gate_values_keep_32_bits(gpu, kind, ff, r, T):
    out_t = r % 32 == 0
    d, rng = 640, np.random.default_rng(T + r)
    u = [np.eye(d, dtype=np.float32)[:, rng.permutation(d)[:r]] for _ in range(2)]
    v = [inputs.random_matrix(rng, r, ff) for _ in range(2)]
    xt = torch.from_numpy(rng.normal(size=(T, d)).astype(np.float32)).to(gpu, torch.bfloat16)
    mats = [torch.from_numpy(np.ascontiguousarray(a)) for a in (u[0], v[0], u[1], v[1])]
    if kind == "fp8":
        q = [fp8.quantize_per_channel(a) for a in mats]
        wide = [torch.from_numpy(O.e4m3_decode(a.data.view(torch.uint8).numpy()) * a.scale.numpy()) for a in q]
        ft = [ops.QuantizedFactor(a.data.to(gpu), a.scale.to(gpu)) for a in q]
        wide[0], wide[2] = mats[0], mats[2]
    else:
        ft = [a.to(gpu, torch.bfloat16) for a in mats]
        wide = [a.float().cpu() for a in ft]
        if kind == "linear":
            ft = [a.t().contiguous().t() for a in ft]
    x64, (ug, vg, uu, vu) = xt.double().cpu(), (a.double() for a in wide)
    g = (x64 @ ug) @ vg
    want = g * torch.sigmoid(g) * ((x64 @ uu) @ vu)
    h = ops.fused_gate_up(xt, *ft, out_transposed=True).t() if out_t else ops.fused_gate_up(xt, *ft)
    err = float((h.cpu().double() - want).norm())
    assert err < 1.05 * float((want.bfloat16().double() - want).norm())


_NW4_CHILD = """
import sys, numpy as np, torch
sys.path[:0] = sys.argv[1].split("|")
from svdmlp import fp8, inputs, ops
x, f = inputs.make_layer(inputs.LayerShape(*map(int, sys.argv[2:6])), T=int(sys.argv[6]), seed=5)
t = [inputs.to_torch(inputs.as_float32(a, torch.bfloat16), torch.bfloat16, torch.device("cuda:0")) for a in (x, *f)]
if int(sys.argv[7]):
    t = t[:1] + [fp8.quantize_per_channel(a) for a in t[1:]]
np.save(sys.argv[8], ops.svd_mlp(*t).view(torch.int16).cpu().numpy())
"""


# The 4-wave tiles (SVDMLP_TUNE=nw=4) have no rank-map instance: such ranks run
# with 8 waves, to the bits of the default.  kg=0: 256-row tiles everywhere, so
# that the 256-wide store stages are reached.
@pytest.mark.parametrize("q", [0, 1])
def test_ranks_off_the_stages_with_four_wave_tiles(gpu, tmp_path, q):
    import os
    import subprocess
    import sys

    got = []
    for tune in ("nw=4,kg=0", "kg=0"):
        out = tmp_path / f"{tune}.npy"
        subprocess.run([sys.executable, "-c", _NW4_CHILD, "|".join(p for p in sys.path if p), "1024", "2048", "1136", "496",
                        "600", str(q), str(out)], env=dict(os.environ, SVDMLP_TUNE=tune), check=True, timeout=120)
        got.append(np.load(out))
    assert np.array_equal(*got)
