"""fp32 attention on the bf16 matrix cores (operands as three bf16 planes) against float64.

Shapes at the edges of the 32-row tiles and 128-row blocks, one to four ranges per key block, padded
widths, both masks with Sq != Sk, zero and negative scales, and operands of very different sizes.  The
planes hold an fp32 value exactly and the kept products leave out less than 2^-24 of each, so the bar is
the fp32 one, 1e-5 max-abs for unit-variance operands (measured: 3e-7 to 3e-6).
"""

import ctypes
import math

import pytest
import torch

from oracle import pe_oracle as O
from pe_ablations_amd import _lib
from pe_ablations_amd.functional import pe_attention
from tests._cmp import err

pytestmark = pytest.mark.gpu


def case(B, Hq, Hkv, Sq, Sk, D, Dv, causal, scale, seed=0, mul=1.0):
    g = torch.Generator().manual_seed(seed + Sq)
    x = {n: torch.randn(B, H, S, d, generator=g) * m for n, H, S, d, m in
         (("q", Hq, Sq, D, mul), ("k", Hkv, Sk, D, 1 / mul), ("v", Hkv, Sk, Dv, 1.0))}
    return x, torch.randn(B, Hq, Sq, Dv, generator=g)


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,Dv,causal,scale", [
    (1, 1, 1, 1, 1, 64, 64, "top_left", 0.125),          # one row
    (1, 2, 1, 33, 33, 40, 48, "top_left", 0.1),          # a tile and a row, padded widths
    (2, 4, 2, 129, 129, 128, 64, "top_left", 0.08),      # a block and a row
    (1, 8, 2, 260, 260, 64, 128, "none", 0.125),         # four ranges of 36 tiles
    (1, 4, 4, 600, 600, 128, 128, "top_left", 0.08),     # ranges that end inside a head
    (1, 2, 1, 100, 355, 256, 128, "bottom_right", 0.06), # QK width 256, Sq < Sk
    (1, 3, 3, 290, 290, 200, 96, "top_left", 0.07),      # 256 padded from 200, 128 from 96
    (1, 2, 2, 70, 70, 64, 64, "top_left", 0.0),          # every visible key alike
    (1, 2, 2, 70, 70, 64, 64, "top_left", -0.1),
])
def test_matches_float64(cuda, B, Hq, Hkv, Sq, Sk, D, Dv, causal, scale):
    x, dout = case(B, Hq, Hkv, Sq, Sk, D, Dv, causal, scale)
    leaves = [x[n].to(cuda).requires_grad_() for n in "qkv"]
    ref_leaves = [x[n].double().requires_grad_() for n in "qkv"]
    out, lse = pe_attention(*leaves, mode="none", scale=scale, causal=False if causal == "none" else causal, return_lse=True)
    ref, rlse = O.attention(*ref_leaves, scale, causal != "none")
    grads = torch.autograd.grad(out, leaves, dout.to(cuda))
    rgrads = torch.autograd.grad(ref, ref_leaves, dout.double())
    assert err(out, ref) < 1e-5 and err(lse, rlse) < 1e-5
    for a, r in zip(grads, rgrads):
        assert err(a, r) < 1e-5 * max(1.0, r.abs().max().item() / 4)


@pytest.mark.parametrize("mul", [1e-12, 1e12])
def test_far_apart_magnitudes(cuda, mul):
    """q and k of sizes whose product is of order one: the planes scale with their operand."""
    x, dout = case(1, 2, 2, 150, 150, 64, 64, "top_left", 0.125, mul=mul)
    leaves = [x[n].to(cuda).requires_grad_() for n in "qkv"]
    ref_leaves = [x[n].double().requires_grad_() for n in "qkv"]
    out = pe_attention(*leaves, mode="none", scale=0.125)
    ref, _ = O.attention(*ref_leaves, 0.125, True)
    assert err(out, ref) < 1e-5
    for a, r in zip(torch.autograd.grad(out, leaves, dout.to(cuda)), torch.autograd.grad(ref, ref_leaves, dout.double())):
        assert err(a, r) < 1e-5 * r.abs().max().item()


def test_a_row_with_one_visible_key(cuda):
    """The first row's output is its value and its lse its score."""
    x, _ = case(1, 1, 1, 64, 64, 64, 64, "bottom_right", 0.125)
    out, lse = pe_attention(*(x[n].to(cuda) for n in "qkv"), mode="none", scale=0.125, causal="bottom_right", return_lse=True)
    assert err(out[0, 0, 0], x["v"][0, 0, 0]) < 1e-6
    assert abs(lse[0, 0, 0].item() - 0.125 * (x["q"][0, 0, 0].double() @ x["k"][0, 0, 0].double()).item()) < 1e-5


def test_noalloc_takes_fp32_calls_that_fit_only_as_fp32_operands(cuda):
    """10000 rows of 4 heads of 128: 153 MB of q~, k~ and v as planes, 102 MB as fp32; the scratch holds
    134 MB.  The no-alloc forward runs such a call on the fp32 unit."""
    from tests.test_zz_no_alloc import _case, _run
    from pe_ablations_amd.functional import _params
    L = _lib.lib()
    q, k, v, freqs, delta, cfg = _case(cuda, 1, 4, 10000, 128, 5, dtype=torch.float32)
    p = _params(cfg, q, k, v, None, delta)
    assert L.pe_attn_fwd_workspace_bytes(ctypes.byref(p)) > L.pe_attn_noalloc_scratch_bytes()
    rc0, out0, lse0 = _run(L, cuda, q, k, v, freqs, delta, cfg, noalloc=False)
    rc1, out1, lse1 = _run(L, cuda, q, k, v, freqs, delta, cfg, noalloc=True)
    assert rc0 == 0 and rc1 == 0
    assert (out0 - out1).abs().max() < 1e-5 and (lse0 - lse1).abs().max() < 1e-5
    assert math.isfinite(out1.sum().item())


@pytest.mark.parametrize("D,Dv,causal", [(64, 64, True), (128, 64, False), (256, 128, True), (40, 48, True)])
def test_infinite_operands(cuda, D, Dv, causal):
    """Infinities in the values, a key and the output's gradient, against the fp32 unit (which an explicit mask
    selects): out, lse and dv infinite, NaN and finite at the same places.  (Whole tiles: the two fill a tile's
    missing rows differently, and 0 times an infinity there is NaN.)"""
    x, dout = case(1, 2, 2, 96, 96, D, Dv, "top_left", 0.1, seed=3)
    x["v"][0, 0, 5, 3], x["v"][0, 0, 40, 7], x["v"][0, 1, 0, 1] = math.inf, -math.inf, math.inf
    x["q"][0, :, :, 2] = x["q"][0, :, :, 2].abs() + 0.1
    x["k"][0, 1, 50, 2] = -math.inf  # never attended to: q there is positive
    dout[0, 0, 60, 9], dout[0, 1, 95, 0] = -math.inf, math.inf
    res = []
    for mask in (None, torch.ones(1, 1, 1, 96, dtype=torch.bool, device=cuda)):
        leaves = [x[n].to(cuda).requires_grad_() for n in "qkv"]
        out, lse = pe_attention(*leaves, mode="none", scale=0.1, causal=causal, mask=mask, return_lse=True)
        res.append((out, lse, torch.autograd.grad(out, leaves[2], dout.to(cuda))[0]))
    for a, b in zip(*res):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf()) and torch.equal(a[a.isinf()], b[b.isinf()])
        fin = b.isfinite()
        assert fin.any() and (a - b)[fin].abs().max() < 2e-5
    assert res[0][0].isinf().any() and res[0][2].isinf().any()


def test_values_at_the_ends_of_the_range(cuda):
    """The largest finite values, whose bf16 rounding is infinite, and small ones.  Of an operand below
    2^-109 the planes hold what is at least 2^-134 of it (half the smallest bf16 subnormal)."""
    q = torch.zeros(1, 1, 64, 64, device=cuda)
    v = torch.full((1, 1, 64, 64), torch.finfo(torch.float32).max, device=cuda)
    v[..., 1::2] *= -1.0
    out = pe_attention(q, q, v, mode="none", scale=0.1, causal="top_left")
    assert torch.equal(out[0, 0, 0], v[0, 0, 0])  # one key: its value
    g = torch.Generator(device=cuda).manual_seed(2)
    q, k, v = (torch.randn(1, 1, 64, 64, generator=g, device=cuda) for _ in range(3))
    for e in (-100, -110, -116, -120):
        out = pe_attention(q, k, v * 2.0 ** e, mode="none", scale=0.1)
        ref, _ = O.attention(q.cpu().double(), k.cpu().double(), (v * 2.0 ** e).cpu().double(), 0.1, True)
        d = (out.cpu().double() - ref).abs().max().item()
        assert d < 1e-5 * 2.0 ** e + 2.0 ** -133
