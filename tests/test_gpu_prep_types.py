"""The vectorised PoPE prologue and dO pass in every element type against their one-wave-per-row forms.

A view whose rows start at an odd element takes the scalar kernels, an aligned one the 16-byte ones; both
evaluate each element alike, so out and lse of the two are bitwise equal.  Shapes take each of the prologue's
launches (small: both sides in one; few heads and a ragged group of eight; a content part in another type
than the rows; padded widths; keys too few for the two-sided launch).  The dO pass sums its rows in another
order in the two forms; Di is a sum of Dv products of unit variance, so the gradients agree to a few
roundings of the compute type.
"""

import math

import pytest
import torch

from pe_ablations_amd.functional import pe_attention

pytestmark = pytest.mark.gpu

H16, B16, F32 = torch.float16, torch.bfloat16, torch.float32


def off_by_one(t):
    """The values of t in a view whose rows start one element past a 16-byte boundary."""
    b, h, s, d = t.shape
    buf = torch.empty(b * s * h * (d + 8) + 8, dtype=t.dtype, device=t.device)
    v = buf[1:1 + b * s * h * (d + 8)].view(b, s, h, d + 8)[..., :d].transpose(1, 2)
    v.copy_(t)
    return v


@pytest.mark.parametrize("xt,ct,B,Hq,Hkv,S,Dc,Dr,Dv,ctype", [
    (H16, H16, 1, 2, 2, 130, 0, 64, 64, None),       # small: one launch for both sides
    (F32, F32, 2, 3, 1, 257, 64, 32, 64, F32),       # split form
    (F32, F32, 2, 9, 9, 1100, 0, 64, 64, None),      # one launch, heads not a multiple of eight
    (H16, H16, 3, 12, 4, 999, 0, 128, 128, None),
    (F32, B16, 2, 8, 4, 500, 64, 32, 64, B16),       # fp32 rows (RMS-normed), bf16 content and compute
    (F32, H16, 4, 10, 10, 700, 0, 64, 64, None),
    (H16, H16, 2, 8, 8, 900, 32, 48, 128, H16),      # 128 columns of 256 are padding's share and content's
    (F32, B16, 1, 1, 1, 8, 0, 16, 64, None),         # fewer keys than the two-sided launch takes
])
def test_vector_rows_equal_scalar_rows(cuda, xt, ct, B, Hq, Hkv, S, Dc, Dr, Dv, ctype):
    g = torch.Generator(device="cuda").manual_seed(S)

    def rows(H, D, dt):
        return torch.randn(B, S, H, D, generator=g, device="cuda").to(dt).transpose(1, 2)

    q, k, v = rows(Hq, Dr, xt), rows(Hkv, Dr, xt), rows(Hkv, Dv, ct)
    qc, kc = (rows(Hq, Dc, ctype), rows(Hkv, Dc, ctype)) if Dc else (None, None)
    freqs = 10000.0 ** (-(torch.arange(0, Dr, dtype=F32, device="cuda") / Dr))
    delta = torch.rand(Hkv, Dr, generator=g, device="cuda") * (-2 * math.pi)
    dout = rows(Hq, Dv, ct)
    got = []
    for move in (lambda t: t, off_by_one):
        leaves = [move(t).detach().requires_grad_() for t in (q, k)]
        out, lse = pe_attention(*leaves, v, q_c=qc, k_c=kc, freqs=freqs, delta=delta, compute_dtype=ct, return_lse=True,
                                start_pos_q=5, start_pos_k=5)
        grads = torch.autograd.grad(out, leaves, move(dout))
        got.append((out, lse, grads))
    (o0, l0, g0), (o1, l1, g1) = got
    assert torch.equal(o0, o1) and torch.equal(l0, l1)
    # one rounding of the 16-bit type where it lands on another side, or a few of fp32's sums
    eps = {F32: 2e-6, H16: 2 ** -9, B16: 2 ** -6}[ct]
    for a, b in zip(g0, g1):
        assert (a.float() - b.float()).abs().max() <= eps * b.float().abs().max()
