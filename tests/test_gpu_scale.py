"""Score factors of zero and below in the 16-bit kernels, against the oracle: the forward, the dK/dV and dQ
kernels of every width (masked tiles at the diagonal and at the end of the keys), the explicit-mask
instantiations, one decoded token and a chunk of new rows.  A negative factor makes the smallest raw score
the likeliest key; 0 makes every visible key alike.  Bars as for positive factors: 2e-2 (bf16) and 2.5e-3
(fp16) max-abs on out and gradients, relative to the largest value where that is above one, 2e-3 on lse.
"""

import pytest
import torch

from oracle import pe_oracle as O
from pe_ablations_amd.functional import cache_widths, pe_attention, pe_attention_decode, pe_cache_append
from tests._cmp import err

pytestmark = pytest.mark.gpu

BAR = {torch.bfloat16: 2e-2, torch.float16: 2.5e-3}


@pytest.mark.parametrize("scale", [0.0, -0.06, 0.06])
@pytest.mark.parametrize("dt,Hq,Hkv,S,D,Dv,masked", [
    (torch.bfloat16, 4, 2, 300, 128, 64, False),
    (torch.bfloat16, 2, 2, 150, 64, 64, False),    # the one-wave dK/dV kernel
    (torch.float16, 2, 1, 333, 256, 128, False),   # QK width 256, split over query ranges
    (torch.bfloat16, 2, 2, 2100, 128, 128, False),  # 96-key tiles
    (torch.bfloat16, 2, 2, 200, 128, 128, True),
    (torch.float16, 2, 2, 130, 64, 64, True),      # the generic gradient kernels
])
def test_training_step(cuda, scale, dt, Hq, Hkv, S, D, Dv, masked):
    g = torch.Generator().manual_seed(S)
    x = [torch.randn(1, H, S, d, generator=g).to(dt) for H, d in ((Hq, D), (Hkv, D), (Hkv, Dv), (Hq, Dv))]
    mask = (torch.arange(S) < S - 40).view(1, 1, 1, S) if masked else None
    leaves, ref_leaves = [t.to(cuda).requires_grad_() for t in x[:3]], [t.double().requires_grad_() for t in x[:3]]
    out, lse = pe_attention(*leaves, mode="none", scale=scale, causal=True, return_lse=True,
                            mask=None if mask is None else mask.to(cuda))
    ref, rlse = O.attention(*ref_leaves, scale, True, mask=mask)
    assert err(out, ref) < BAR[dt] and err(lse, rlse) < 2e-3
    grads = torch.autograd.grad(out, leaves, x[3].to(cuda))
    rgrads = torch.autograd.grad(ref, ref_leaves, x[3].double())
    for a, r in zip(grads, rgrads):
        assert err(a, r) < BAR[dt] * max(1.0, r.abs().max().item())


@pytest.mark.parametrize("scale", [0.0, -0.06])
@pytest.mark.parametrize("dt,Hq,Hkv,L,Sq,D,Dv", [
    (torch.bfloat16, 4, 2, 333, 1, 128, 64),       # one decoded token
    (torch.bfloat16, 10, 10, 700, 64, 128, 128),   # chunks: 128-row blocks
    (torch.float16, 6, 2, 777, 257, 256, 128),     # 256-row blocks, QK width 256
    (torch.bfloat16, 2, 2, 500, 400, 64, 64),      # key tiles cut by the diagonal and the cache's end
])
def test_cache(cuda, scale, dt, Hq, Hkv, L, Sq, D, Dv):
    g = torch.Generator().manual_seed(L)
    q, k, v = (torch.randn(1, H, n, d, generator=g).to(dt) for H, n, d in ((Hq, Sq, D), (Hkv, L, D), (Hkv, L, Dv)))
    wk, wv = cache_widths(mode="none", d_pe=D, d_v=Dv)
    kc, vc = (torch.full((1, Hkv, L + 9, w), float("nan"), dtype=dt, device=cuda) for w in (wk, wv))
    pe_cache_append(k.to(cuda), v.to(cuda), kc, vc, start_pos=0, mode="none")
    with torch.no_grad():
        out, lse = pe_attention_decode(q.to(cuda), kc, vc, L, d_v=Dv, mode="none", scale=scale, return_lse=True)
    ref, rlse = O.attention(q.float(), k.float(), v.float(), scale, causal=True)
    assert err(out, ref) < BAR[dt] and err(lse, rlse) < 2e-3
