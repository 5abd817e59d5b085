"""The fused RMSNorm + PoPE prologue of both sides in one launch against the norm (pe_rmsnorm_fwd) followed by
the unfused prologue, which round every element alike: out and lse are bitwise equal.  Widths whose chunks
divide a wave (one set of phases per lane) and do not (24 dims), shared and per-head phase biases, more query
than key features, content parts and every compute type.
"""

import math

import pytest
import torch

from pe_ablations_amd.functional import pe_attention, rms_norm

pytestmark = pytest.mark.gpu
F32, B16, H16 = torch.float32, torch.bfloat16, torch.float16


@pytest.mark.parametrize("dt,B,Hq,Hkv,S,Dc,Dr,Dv,per_head", [
    (B16, 2, 8, 4, 70, 64, 32, 64, False),
    (B16, 1, 16, 16, 33, 0, 128, 128, True),
    (H16, 1, 6, 2, 129, 0, 64, 64, True),
    (F32, 2, 4, 4, 65, 32, 24, 64, False),
    (F32, 1, 3, 1, 5, 0, 64, 64, False),
    (B16, 1, 32, 2, 40, 64, 32, 64, True),
])
def test_fused_equals_norm_then_prologue(cuda, dt, B, Hq, Hkv, S, Dc, Dr, Dv, per_head):
    g = torch.Generator(device="cuda").manual_seed(S)

    def rows(H, D):
        return torch.randn(B, S, H * D, generator=g, device="cuda").to(dt)

    def heads(t, H):
        return t.view(B, S, H, -1).transpose(1, 2)

    q, k, v = rows(Hq, Dr), rows(Hkv, Dr), heads(rows(Hkv, Dv), Hkv)
    c = dict(q_c=heads(rows(Hq, Dc), Hq), k_c=heads(rows(Hkv, Dc), Hkv)) if Dc else {}
    wq, wk = ((1 + 0.1 * torch.randn(H * Dr, generator=g, device="cuda")).to(dt) for H in (Hq, Hkv))
    freqs = 10000.0 ** (-(torch.arange(0, Dr, dtype=F32, device="cuda") / Dr))
    delta = torch.rand((Hkv, Dr) if per_head else (Dr,), generator=g, device="cuda") * (-2 * math.pi)
    kw = dict(freqs=freqs, delta=delta, return_lse=True, start_pos_q=7, start_pos_k=7, **c)
    with torch.no_grad():
        a = pe_attention(heads(q, Hq), heads(k, Hkv), v, qr_norm_weight=wq, kr_norm_weight=wk, **kw)
        b = pe_attention(heads(rms_norm(q, wq), Hq), heads(rms_norm(k, wk), Hkv), v, **kw)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
