"""The RoPE / no-PE prologue over several heads and the gradient fused into the dQ and dK/dV epilogues, at
head widths 64 and 128, against the stand-alone kernels: views whose rows start at an odd element take those,
aligned ones the fused path, and both evaluate every element alike, so out, dq, dk and dv are bitwise equal.
Shapes: heads not a multiple of the prologue's group, rows past the last full block, a key-block list shared
out over workgroups (S > 512), and key positions that start elsewhere than the queries' (no shared angles).
"""

import pytest
import torch

from pe_ablations_amd.functional import pe_attention
from tests.test_gpu_prep_types import off_by_one

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,dt,B,Hq,Hkv,S,D,norm,start_k", [
    ("rope", torch.bfloat16, 1, 5, 5, 130, 128, True, 3),
    ("rope", torch.float16, 2, 6, 2, 257, 128, False, 3),
    ("rope", torch.bfloat16, 1, 4, 2, 600, 128, True, 3),
    ("rope", torch.bfloat16, 1, 3, 1, 200, 128, True, 40),
    ("none", torch.bfloat16, 1, 4, 4, 300, 128, True, 3),
    ("rope", torch.float16, 1, 9, 3, 333, 64, True, 3),
    ("rope", torch.bfloat16, 1, 2, 2, 1, 128, False, 3),
])
def test_fused_equals_stand_alone(cuda, mode, dt, B, Hq, Hkv, S, D, norm, start_k):
    g = torch.Generator(device="cuda").manual_seed(S)
    q, k, v, dout = (torch.randn(B, S, H, D, generator=g, device="cuda").to(dt).transpose(1, 2) for H in (Hq, Hkv, Hkv, Hq))
    freqs = 10000.0 ** (-(torch.arange(0, D, 2, dtype=torch.float32, device="cuda") / D)) if mode == "rope" else None
    got = []
    for move in (lambda t: t, off_by_one):
        leaves = [move(t).detach().requires_grad_() for t in (q, k)] + [v.detach().requires_grad_()]
        out = pe_attention(*leaves, mode=mode, freqs=freqs, qk_norm=norm, start_pos_q=3, start_pos_k=start_k)
        got.append([out] + list(torch.autograd.grad(out, leaves, dout)))
    for a, b in zip(*got):
        assert torch.equal(a, b)
