"""The dK/dV kernel with each key block's (query head, query tile) list shared out over workgroups: ranges
that end inside a head and inside a 64-query tile pair, ranges of the last key block with fewer tiles than
ranges, and both masks, against the oracle in fp64 on the operands as given (no positional transform).

Bars as in the random sweep: 2e-2 (bf16) and 2.5e-3 (fp16) max-abs, scaled by a quarter of the largest
value above magnitude 4.
"""

import pytest
import torch

from oracle import pe_oracle as O
from pe_ablations_amd.functional import pe_attention
from tests._cmp import err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,B,Hq,Hkv,Sq,Sk,D,Dv,causal", [
    ("bf16", 1, 1, 1, 513, 513, 128, 64, True),            # 64-query tiles, two ranges of each block
    ("bf16", 1, 3, 1, 700, 700, 128, 128, True),           # three heads: ranges cross from one to the next
    ("fp16", 1, 2, 2, 1025, 1025, 128, 64, True),          # 32-query tiles, last block with one tile
    ("bf16", 1, 4, 2, 600, 777, 256, 128, "bottom_right"),
    ("bf16", 2, 2, 1, 530, 530, 256, 64, False),
    ("fp16", 1, 4, 1, 640, 640, 200, 96, True),            # padded widths
    ("bf16", 1, 16, 1, 2001, 2001, 128, 64, True),         # sixteen ranges, last block with as many tiles
    ("fp16", 1, 64, 1, 520, 1000, 128, 128, "bottom_right"),  # sixteen ranges of four heads
])
def test_ranges_match_oracle(cuda, dtype, B, Hq, Hkv, Sq, Sk, D, Dv, causal):
    dt = torch.bfloat16 if dtype == "bf16" else torch.float16
    g = torch.Generator().manual_seed(Sq)
    x = [torch.randn(B, H, S, d, generator=g).to(dt) for H, S, d in ((Hq, Sq, D), (Hkv, Sk, D), (Hkv, Sk, Dv))]
    dout = torch.randn(B, Hq, Sq, Dv, generator=g).to(dt)
    leaves = [t.to(cuda).requires_grad_() for t in x]
    out = pe_attention(*leaves, mode="none", scale=D ** -0.5, causal=causal)
    grads = torch.autograd.grad(out, leaves, dout.to(cuda))
    again = torch.autograd.grad(pe_attention(*leaves, mode="none", scale=D ** -0.5, causal=causal), leaves, dout.to(cuda))
    ref_leaves = [t.double().requires_grad_() for t in x]
    ref, _ = O.attention(*ref_leaves, D ** -0.5, causal is not False)
    base = 2e-2 if dt == torch.bfloat16 else 2.5e-3
    for a, b, r in zip(grads, again, torch.autograd.grad(ref, ref_leaves, dout.double())):
        assert torch.equal(a, b)  # the partials are added in a fixed order
        assert err(a, r) < base * max(1.0, r.abs().max().item() / 4), err(a, r)
