"""fp32 attention as split products (three bf16 planes per value): parity at the edges of its range, precision against
the fp64 oracle, and non-finite and huge inputs, which it hands to the fp32 MFMA."""

import math

import pytest
import torch

import oracle
from ebr_amd.fused_attn import ops

pytestmark = pytest.mark.gpu
F32 = torch.float32

# L around the 32-row chunks, the 64-row blocks and the 128-row border of the one-workgroup kernels; D below, at and
# above the 32- and 64-wide instances; one shape each where the rule falls back to the fp32 MFMA (L = 128, D = 64; D = 16)
SHAPES = [(1, 2, 33, 32), (1, 2, 64, 20), (2, 1, 97, 32), (1, 1, 128, 32), (1, 2, 129, 32), (2, 2, 129, 64),
          (1, 1, 160, 36), (1, 2, 193, 128), (1, 1, 257, 100), (1, 1, 320, 64), (1, 1, 128, 64), (1, 1, 130, 16)]


def _run(q, k, v, do, gq, gk, gv, scale):
    o, lse = ops._hip_fwd(q, k, v, scale)
    d = ops._hip_bwd(q, k, v, o, lse, do, scale)
    return [o, lse, *d, *ops._hip_bwd_bwd(q, k, v, o, lse, do, gq, gk, gv, scale)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("views", [False, True])
def test_against_the_oracle_in_64_bits(shape, views):
    B, H, L, D = shape
    ts = oracle.make_inputs(B, H, L, D, dtype=F32, seed=L + D, qkv_scale=0.7)
    dev = [t.cuda() for t in ts]
    if views:  # rows of a [B, L, 3 H D] projection
        qkv = torch.stack(dev[:3], dim=0).permute(1, 3, 0, 2, 4).contiguous()
        dev[:3] = [qkv[:, :, i].transpose(1, 2) for i in range(3)]
    scale = D**-0.5
    got = _run(*dev, scale)
    q, k, v, do, gq, gk, gv = (t.double() for t in ts)
    o, lse = oracle.attn_fwd(q, k, v, scale)
    want = [o, lse, *oracle.attn_bwd(q, k, v, o, lse, do, scale),
            *oracle.attn_bwd_bwd(q, k, v, o, lse, do, None, gq, gk, gv, scale)]
    for a, r in zip(got, want):
        a = a.double().cpu()
        # fp32 sums of up to L terms, lse and P rounded to 2^-24: the fp32 MFMA shows 7e-7 at L = 400
        assert ((a - r).norm() / r.norm()).item() < 1.5e-6
        assert oracle.rel_err(a, r) < 1e-5


@pytest.mark.parametrize("shape", [(1, 2, 140, 64), (1, 1, 50, 32)])
def test_non_finite_and_huge_values_as_in_fp32(shape):
    B, H, L, D = shape
    q, k, v, do, gq, gk, gv = (t.cuda() for t in oracle.make_inputs(B, H, L, D, dtype=F32, seed=1, qkv_scale=0.5))
    scale = D**-0.5
    v2 = v.clone()
    v2[0, 0, 3, 5] = float("inf")
    v2[0, 0, 9, 7] = 3.4e38  # past the largest bf16
    v2[0, 0, 11, 8] = float("nan")
    o, _ = ops._hip_fwd(q, k, v2, scale)
    p = torch.softmax(q.cpu() @ k.cpu().transpose(-1, -2) * scale, dim=-1)
    want = p @ v2.cpu()
    assert torch.equal(torch.isinf(o.cpu()), torch.isinf(want)) and torch.equal(torch.isnan(o.cpu()), torch.isnan(want))
    fine = torch.isfinite(want)
    torch.testing.assert_close(o.cpu()[fine], want[fine], rtol=1e-5, atol=1e-5)
    # dV = P^T dO column by column: an infinite dO entry stays in its column
    o, lse = ops._hip_fwd(q, k, v, scale)
    do2 = do.clone()
    do2[0, 0, 2, 4] = float("inf")
    _, _, dv = ops._hip_bwd(q, k, v, o, lse, do2, scale)
    want = p.transpose(-1, -2) @ do2.cpu()
    assert torch.equal(torch.isinf(dv.cpu()), torch.isinf(want)) and not torch.isnan(dv).any()
    fine = torch.isfinite(want)
    torch.testing.assert_close(dv.cpu()[fine], want[fine], rtol=1e-5, atol=1e-5)
    # one in the backward of the backward's cotangent: hV's and hdO's columns as in fp32 arithmetic
    gv2 = gv.clone()
    gv2[0, 0, 6, 1] = float("inf")
    hdo = ops._hip_bwd_bwd(q, k, v, o, lse, do, gq, gk, gv2, scale)[3].cpu()
    assert torch.isinf(hdo[0, 0, :, 1]).all() and torch.isfinite(hdo[0, 0, :, 2:]).all()


@pytest.mark.parametrize("shape", [(1, 2, 140, 64), (1, 1, 50, 32)])
@pytest.mark.parametrize("size", [1e-30, 1e-36])
def test_tiny_values_keep_their_precision(shape, size):
    """Values whose smaller parts fall below bf16's normal range: fp32 carries them, and so does the op."""
    B, H, L, D = shape
    q, k, v, do, gq, gk, gv = (t.cuda() for t in oracle.make_inputs(B, H, L, D, dtype=F32, seed=2, qkv_scale=0.5))
    scale = D**-0.5
    o, lse = ops._hip_fwd(q, k, v * size, scale)
    p = torch.softmax(q.cpu().double() @ k.cpu().double().transpose(-1, -2) * scale, dim=-1)
    want = p @ (v * size).cpu().double()
    assert ((o.cpu().double() - want).norm() / want.norm()).item() < 1.5e-6
    o, lse = ops._hip_fwd(q, k, v, scale)
    dv = ops._hip_bwd(q, k, v, o, lse, do * size, scale)[2].cpu().double()
    want = p.transpose(-1, -2) @ (do * size).cpu().double()
    assert ((dv - want).norm() / want.norm()).item() < 1.5e-6


SCALED = {  # powers of two on q, k, v, dO, gQ, gK, gV that leave the probabilities as they are
    "small dO against large k": (-20, 20, 0, -118, -20, 20, 0),
    "small q against large k": (-118, 118, 0, 0, -118, 118, 0),
    "small v against large dO": (0, 0, -118, 118, 0, 0, -118),
    "small cotangents": (0, 0, 0, 0, -118, -118, -118),
}


@pytest.mark.parametrize("shape", [(1, 2, 140, 64), (1, 1, 50, 32), (1, 1, 130, 128)])
@pytest.mark.parametrize("powers", SCALED.values(), ids=SCALED.keys())
def test_every_output_keeps_its_precision_on_scaled_operands(shape, powers):
    """Operands near 2^-126 (a plane of unscaled remainders would lose their low bits) beside ones that make up for it:
    the sums and the outputs are ordinary numbers, so their size says nothing about the operands."""
    B, H, L, D = shape
    ts = oracle.make_inputs(B, H, L, D, dtype=F32, seed=3, qkv_scale=0.7)
    ts = [t * 2.0**p for t, p in zip(ts, powers)]
    scale = D**-0.5
    got = _run(*(t.cuda() for t in ts), scale)
    q, k, v, do, gq, gk, gv = (t.double() for t in ts)
    o, lse = oracle.attn_fwd(q, k, v, scale)
    want = [o, lse, *oracle.attn_bwd(q, k, v, o, lse, do, scale),
            *oracle.attn_bwd_bwd(q, k, v, o, lse, do, None, gq, gk, gv, scale)]
    for name, a, r in zip(("o", "lse", "dq", "dk", "dv", "hq", "hk", "hv", "hdo"), got, want):
        # as on ordinary operands, plus, where an output is subnormal, half a quantum for each of its sums' L terms
        bound = 1.5e-6 * r.norm() + L * 2.0**-150 * r.numel() ** 0.5
        assert (a.double().cpu() - r).norm() <= bound, name


@pytest.mark.parametrize("shape", [(1, 2, 140, 64), (1, 1, 50, 32)])
def test_scores_that_overflow_only_before_the_scale(shape):
    """Sums of q k around -2^96, where the planes' own scale overflows some of a row's, with a scale that makes ordinary
    scores of them."""
    B, H, L, D = shape
    q, k, v, do, gq, gk, gv = oracle.make_inputs(B, H, L, D, dtype=F32, seed=5, qkv_scale=0.7)
    q, k = q.abs(), -k.abs()
    q = q * -(2.0**48 / (q @ k.transpose(-1, -2)).mean(-1, keepdim=True))  # a row's scores lie around -2^48 of k's unit
    k, gq, gk = k * 2.0**48, gq * 2.0**48, gk * 2.0**48
    ts, scale = (q, k, v, do, gq, gk, gv), 2.0**-92
    s = q.double() @ k.double().transpose(-1, -2)
    assert (s < -(2.0**96)).any(-1).all() and (s > -(2.0**96)).any(-1).all()  # every row has scores on either side
    got = _run(*(t.cuda() for t in ts), scale)
    q, k, v, do, gq, gk, gv = (t.double() for t in ts)
    o, lse = oracle.attn_fwd(q, k, v, scale)
    want = [o, lse, *oracle.attn_bwd(q, k, v, o, lse, do, scale),
            *oracle.attn_bwd_bwd(q, k, v, o, lse, do, None, gq, gk, gv, scale)]
    # scores of about -16, each rounded to 2^-24 of itself before the exponential
    for name, a, r in zip(("o", "lse", "dq", "dk", "dv", "hq", "hk", "hv", "hdo"), got, want):
        assert (a.double().cpu() - r).norm() <= 16 * 2.0**-22 * r.norm(), name


def test_repeated_calls_give_the_same_bits():
    ts = [t.cuda() for t in oracle.make_inputs(2, 2, 200, 64, dtype=F32, seed=4, qkv_scale=0.5)]
    first = _run(*ts, 0.125)
    for a, b in zip(first, _run(*ts, 0.125)):
        assert torch.equal(a, b)
