"""Decode with the query transform inside the split kernel (content part, fp16, padded widths) and with the
ranges merged in the workgroup, against the paths they replace.

A query view whose rows start at an odd element is transformed by the prologue launch, an aligned one in the
kernel, with the same arithmetic: bitwise equal results.  Short caches (see decode_plan in pe_api.cpp) and
those of 256 or more tiles are merged in the workgroup, the others by the merge kernel; all are held to the
oracle at the decode bars.
"""

import math

import pytest
import torch

from oracle import pe_oracle as O
from pe_ablations_amd.functional import cache_widths, pe_attention_decode, pe_cache_append
from tests._cmp import err
from tests.test_gpu_prep_types import off_by_one

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,B,Hq,Hkv,L,Sq,Dc,Dr,Dv", [
    (torch.bfloat16, 1, 8, 4, 500, 1, 64, 32, 64),     # the reference's shape
    (torch.float16, 3, 8, 1, 512, 1, 0, 64, 64),
    (torch.bfloat16, 2, 4, 4, 33, 2, 32, 16, 128),     # padded width, a block and a row
    (torch.float16, 1, 6, 2, 1, 1, 64, 32, 48),        # one row, padded values
    (torch.bfloat16, 1, 2, 1, 513, 4, 0, 128, 128),    # the merge kernel
    (torch.bfloat16, 1, 16, 2, 300, 1, 128, 64, 128),  # QK width 256, eight rows a tile
    (torch.bfloat16, 2, 12, 2, 200, 9, 0, 64, 64),     # 54 rows, two tiles, prologue launch
    (torch.bfloat16, 1, 12, 1, 200, 2, 64, 32, 48),    # 24 rows merged four columns at a time, padded values
    (torch.float16, 1, 10, 2, 90, 7, 0, 128, 128),     # 35 rows: a full tile and three rows
])
def test_decode_matches_oracle_and_the_prologue_launch(cuda, dt, B, Hq, Hkv, L, Sq, Dc, Dr, Dv):
    g = torch.Generator().manual_seed(L)
    x = {n: torch.randn(B, S, H, D, generator=g).to(dt).transpose(1, 2) for n, H, S, D in
         (("q", Hq, Sq, Dr), ("k", Hkv, L, Dr), ("v", Hkv, L, Dv), ("qc", Hq, Sq, Dc), ("kc", Hkv, L, Dc)) if D}
    on = (lambda n: x[n].cuda() if n in x else None)
    Sq = min(Sq, L)
    freqs, delta = O.pope_freqs(Dr), torch.rand(Dr, generator=g) * (-2 * math.pi)
    wk, wv = cache_widths(d_content=Dc, d_pe=Dr, d_v=Dv)
    kc, vc = (torch.full((B, Hkv, L + 5, w), float("nan"), dtype=dt, device=cuda) for w in (wk, wv))
    pe_cache_append(on("k"), on("v"), kc, vc, start_pos=0, k_c=on("kc"), freqs=freqs.cuda(), delta=delta.cuda())
    kw = dict(d_v=Dv, freqs=freqs.cuda(), scale=0.1, return_lse=True)
    with torch.no_grad():
        out, lse = pe_attention_decode(on("q"), kc, vc, L, q_c=on("qc"), **kw)
        out2, lse2 = pe_attention_decode(off_by_one(on("q")), kc, vc, L, q_c=on("qc"), **kw)
    assert torch.equal(out, out2) and torch.equal(lse, lse2)
    tq, tk = O.pope_transform(x["q"], freqs, L - Sq), O.pope_transform(x["k"], freqs, 0, delta)
    if Dc:
        tq, tk = torch.cat([x["qc"].float(), tq], -1), torch.cat([x["kc"].float(), tk], -1)
    ref, rlse = O.attention(tq.to(dt).float(), tk.to(dt).float(), x["v"].float(), 0.1, causal=True)
    assert err(out, ref) < (2e-2 if dt == torch.bfloat16 else 2.5e-3) and err(lse, rlse) < 2e-3


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("step", [0.0, 3.0, 5.9, 6.1, 80.0, -5.0, -80.0])
def test_reference_follows_falling_and_rising_blocks(cuda, dt, step):
    """Short caches whose 32-key blocks' largest scores fall (or rise) by ``step`` powers of two a block.
    Bar: half an ulp for each probability and for the result, so 2^-8 (fp16: 2^-11) of the largest value; lse
    from fp32 sums of magnitudes up to 80 * 16 * ln 2: 2^-21 of that."""
    g = torch.Generator().manual_seed(5)
    L, Hq, Hkv, Dc, Dr, Dv = 512, 4, 2, 64, 32, 64
    qc, kc = torch.zeros(1, Hq, 1, Dc, dtype=dt), torch.zeros(1, Hkv, L, Dc, dtype=dt)
    qc[..., 0] = 8.0
    kc[..., 0] = (-step * math.log(2.0) * (torch.arange(L) // 32) + torch.randn(Hkv, L, generator=g)).to(dt)
    qr = torch.full((1, Hq, 1, Dr), -30.0, dtype=dt)  # softplus 1e-13: the position part adds nothing
    kr, v = torch.randn(1, Hkv, L, Dr, generator=g).to(dt), torch.randn(1, Hkv, L, Dv, generator=g).to(dt)
    freqs, delta = O.pope_freqs(Dr).cuda(), torch.zeros(Dr, device=cuda)
    wk, wv = cache_widths(d_content=Dc, d_pe=Dr, d_v=Dv)
    ck, cv = (torch.zeros(1, Hkv, L, w, dtype=dt, device=cuda) for w in (wk, wv))
    pe_cache_append(kr.cuda(), v.cuda(), ck, cv, start_pos=0, k_c=kc.cuda(), freqs=freqs, delta=delta)
    with torch.no_grad():
        out, lse = pe_attention_decode(qr.cuda(), ck, cv, L, q_c=qc.cuda(), d_v=Dv, freqs=freqs, scale=0.125, return_lse=True)
    s = kc[..., 0].double().repeat_interleave(Hq // Hkv, 1)
    ref = s.softmax(-1).unsqueeze(-2) @ v.double().repeat_interleave(Hq // Hkv, 1)
    assert err(out, ref) < (2 ** -8 if dt == torch.bfloat16 else 2 ** -11) * float(v.abs().max())
    assert err(lse[..., 0], s.logsumexp(-1)) < 2 ** -21 * max(16.0, abs(step) * 16)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("step", [0.0, 4.9, 5.9])
def test_long_caches_of_many_tiles(cuda, dt, step):
    """256 (batch entry, kv head) units leave four ranges each, merged in the workgroup, also for a cache of
    1100 rows: nine blocks a wave, whose scores fall by ``step`` powers of two a block.  Values of 2^114 (not
    in fp16): sums must stay within 2^14 of the largest value.  Bar as above, fp32 sums: 2^-18."""
    g = torch.Generator(device="cuda").manual_seed(7)
    B, Hq, Hkv, L, Dc, Dr, Dv = 32, 16, 8, 1100, 64, 32, 64
    qc, kc = torch.zeros(B, Hq, 1, Dc, dtype=dt, device=cuda), torch.zeros(B, Hkv, L, Dc, dtype=dt, device=cuda)
    qc[..., 0] = 8.0
    kc[..., 0] = (-step * math.log(2.0) * (torch.arange(L, device=cuda) // 32)).to(dt)
    qr = torch.full((B, Hq, 1, Dr), -30.0, dtype=dt, device=cuda)
    kr = torch.zeros(B, Hkv, L, Dr, dtype=dt, device=cuda)
    v = ((1 + torch.rand(B, Hkv, L, Dv, generator=g, device=cuda)) * (1.0 if dt == torch.float16 else 2.0 ** 114)).to(dt)
    freqs = O.pope_freqs(Dr).cuda()
    wk, wv = cache_widths(d_content=Dc, d_pe=Dr, d_v=Dv)
    ck, cv = (torch.zeros(B, Hkv, L, w, dtype=dt, device=cuda) for w in (wk, wv))
    pe_cache_append(kr, v, ck, cv, start_pos=0, k_c=kc, freqs=freqs)
    with torch.no_grad():
        out, lse = pe_attention_decode(qr, ck, cv, L, q_c=qc, d_v=Dv, freqs=freqs, scale=0.125, return_lse=True)
    s = kc[..., 0].double().repeat_interleave(Hq // Hkv, 1)
    ref = s.softmax(-1).unsqueeze(-2) @ v.double().repeat_interleave(Hq // Hkv, 1)
    bar = {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11, torch.float32: 2 ** -18}[dt]
    assert err(out, ref) < bar * float(v.abs().max())
    assert err(lse[..., 0], s.logsumexp(-1)) < 2 ** -21 * max(16.0, abs(step) * 35)
