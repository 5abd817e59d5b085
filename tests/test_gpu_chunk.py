"""Cache attention of many new rows (a prompt prefilled in chunks), which runs the forward kernel over key
ranges of the cache, against the oracle.

The rows of one kv head's query heads follow each other in the kernel's 128- or 256-row blocks, so the
cases put the ends of heads, blocks, key tiles (64 and 96 keys) and key ranges in different places: the
fewest rows that take this path and one more than a block holds, blocks that span several heads, one key
range and many, a cache hardly longer than the chunk, and both masks.  The oracle transforms the rows,
rounds them to the operand type and attends in fp64; bars 2e-2 (bf16) and 2.5e-3 (fp16) max-abs on out,
2e-3 on lse, as for single decoded rows.
"""

import math

import pytest
import torch

from oracle import pe_oracle as O
from pe_ablations_amd.functional import cache_widths, pe_attention_decode, pe_cache_append
from tests._cmp import err, half_ulp_bf16

pytestmark = pytest.mark.gpu

CASES = [  # mode, dtype, B, Hq, Hkv, L, Sq, Dc, Dr, Dv, causal
    ("pope", "bf16", 1, 10, 10, 700, 64, 0, 128, 128, "bottom_right"),  # the fewest rows, one 128-row block
    ("pope", "bf16", 2, 4, 2, 1999, 129, 64, 32, 64, "bottom_right"),   # 258 rows, two heads in a block
    ("pope", "fp16", 1, 6, 2, 777, 257, 0, 64, 64, "bottom_right"),     # 771 rows of three heads
    ("rope", "bf16", 1, 8, 1, 500, 96, 0, 128, 128, "bottom_right"),    # 768 rows, two ranges of keys
    ("pope", "bf16", 1, 16, 2, 6001, 83, 0, 64, 64, "bottom_right"),    # 664 rows, many ranges
    ("none", "fp16", 1, 3, 3, 640, 600, 0, 64, 128, "bottom_right"),    # the first range ends before the diagonal
    ("pope", "bf16", 1, 2, 2, 1100, 321, 0, 128, 64, "none"),           # QK width 256, no mask
    ("pope", "bf16", 1, 1, 1, 1300, 1300, 0, 128, 128, "bottom_right"),  # every row new: rows with one visible key
    ("rope", "bf16", 4, 16, 4, 256, 100, 0, 64, 64, "bottom_right"),     # short caches: the decode kernel, 208 tiles
    ("pope", "bf16", 2, 16, 16, 300, 64, 0, 128, 128, "bottom_right"),   # one range, 2048 rows in all
    ("pope", "fp16", 4, 16, 4, 200, 200, 64, 32, 64, "bottom_right"),    # more tiles than the decode kernel takes at once
]


@pytest.mark.parametrize("mode,dtype,B,Hq,Hkv,L,Sq,Dc,Dr,Dv,causal", CASES)
def test_chunk_matches_oracle(cuda, mode, dtype, B, Hq, Hkv, L, Sq, Dc, Dr, Dv, causal):
    g = torch.Generator().manual_seed(L + Sq)
    dt = torch.bfloat16 if dtype == "bf16" else torch.float16
    k, v = torch.randn(B, Hkv, L, Dr, generator=g).to(dt), torch.randn(B, Hkv, L, Dv, generator=g).to(dt)
    q = torch.randn(B, Hq, Sq, Dr, generator=g).to(dt)
    kc = torch.randn(B, Hkv, L, Dc, generator=g).to(dt) if Dc else None
    qc = torch.randn(B, Hq, Sq, Dc, generator=g).to(dt) if Dc else None
    freqs = delta = None
    if mode == "pope":
        freqs, delta = O.pope_freqs(Dr), torch.rand(Dr, generator=g) * (-2 * math.pi)
    elif mode == "rope":
        freqs = O.rope_inv_freq(Dr)
    on = (lambda t: None if t is None else t.to(cuda))
    wk, wv = cache_widths(mode=mode, d_content=Dc, d_pe=Dr, d_v=Dv)
    # capacity past the length, its rows poisoned: they must not be read
    kcache = torch.full((B, Hkv, L + 37, wk), float("nan"), dtype=dt, device=cuda)
    vcache = torch.full((B, Hkv, L + 37, wv), float("nan"), dtype=dt, device=cuda)
    pe_cache_append(on(k), on(v), kcache, vcache, start_pos=0, mode=mode, k_c=on(kc), freqs=on(freqs), delta=on(delta))
    scale = (Dc + 2 * Dr) ** -0.5 if mode == "pope" else Dr ** -0.5
    with torch.no_grad():
        out, lse = pe_attention_decode(on(q), kcache, vcache, L, d_v=Dv, mode=mode, q_c=on(qc), freqs=on(freqs),
                                       scale=scale, causal=causal, return_lse=True)
    if mode == "pope":
        tq, tk = O.pope_transform(q, freqs, L - Sq), O.pope_transform(k, freqs, 0, delta)
        if Dc:
            tq, tk = torch.cat([qc.float(), tq], -1), torch.cat([kc.float(), tk], -1)
    elif mode == "rope":
        tq, tk = O.rope_rotate(q, freqs, L - Sq), O.rope_rotate(k, freqs, 0)
    else:
        tq, tk = q.float(), k.float()
    ref, rlse = O.attention(tq.to(dt).float(), tk.to(dt).float(), v.float(), scale, causal=causal != "none")
    assert err(out, ref) < (2e-2 if dt == torch.bfloat16 else 2.5e-3), err(out, ref)
    assert err(lse, rlse) < 2e-3, err(lse, rlse)


@pytest.mark.parametrize("dt,Hq,Sq,Dr", [(torch.bfloat16, 4, 300, 64), (torch.float16, 10, 64, 128), (torch.bfloat16, 4, 300, 256)])
def test_the_largest_probability_of_a_tile_is_not_rounded(cuda, dt, Hq, Sq, Dr):
    """Key 150, in a later tile of the first key range, stands x in (0, 7.5] powers of two above all others and
    alone has a value, so out = v 2^x / (2^x + 999): as P is relative to its tile's max, its probability there
    is 1, and all that is left is the result's own rounding, half an ulp (and 2^-18 for exp2 and the fp32 sums)."""
    g = torch.Generator().manual_seed(Sq)
    L, j, Dv = 1000, 150, 64
    x = torch.rand(1, Hq, Sq, generator=g) * 7.5
    q, k, v = torch.zeros(1, Hq, Sq, Dr), torch.zeros(1, Hq, L, Dr), torch.zeros(1, Hq, L, Dv)
    q[..., 0], k[:, :, j, 0] = x, 1.0
    v[:, :, j] = torch.randn(1, Hq, Dv, generator=g)
    q, k, v = q.to(dt), k.to(dt), v.to(dt)
    wk, wv = cache_widths(mode="none", d_pe=Dr, d_v=Dv)
    kcache, vcache = (torch.zeros(1, Hq, L, w, dtype=dt, device=cuda) for w in (wk, wv))
    pe_cache_append(k.to(cuda), v.to(cuda), kcache, vcache, start_pos=0, mode="none")
    with torch.no_grad():
        out = pe_attention_decode(q.to(cuda), kcache, vcache, L, d_v=Dv, mode="none", scale=math.log(2.0), causal=False)
    e = torch.exp2(q[..., :1].double())
    ref = v[:, :, j:j + 1].double() * e / (e + (L - 1))
    half = half_ulp_bf16(ref) if dt == torch.bfloat16 else (half_ulp_bf16(ref) / 8).clamp_min(2.0 ** -25)  # fp16 subnormals
    assert ((out.double().cpu() - ref).abs() <= half + ref.abs() * 2.0 ** -18).all()
