"""The work that users of this package have it do, as cases that can be timed and compared.

A case is a dict of plain values.  Its ``kind`` says which path it takes:

* ``train``   one training step of the fused attention: ``pe_attention`` forward and backward, the
  output and every gradient returned;
* ``eval``    one forward without gradients (long-context evaluation);
* ``decode``  one step of generation on a KV cache: ``pe_cache_append`` of the new rows, then
  ``pe_attention_decode`` of the new queries.  ``Sq`` = 1 is a decoded token; more rows are a chunk
  of a prompt that is prefilled in pieces;
* ``block``   one training step of a whole ``TransformerBlock`` under bf16 autocast with fp32
  weights, as a trainer runs it: output, input gradient and every parameter's gradient.

The listed sizes are the ones the package's own configurations, tests and benchmark use, or
generic; ``draw`` spreads the same kinds over their ranges.
"""

import math

import torch
import torch.nn.functional as F

from pe_ablations_amd.functional import cache_widths, pe_attention, pe_attention_decode, pe_cache_append
from pe_ablations_amd.pope import PoPEEmbedding
from pe_ablations_amd.rope import RotaryEmbedding
from pe_ablations_amd.transformer import TransformerBlock, TransformerConfig

DTYPE = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _attn(name, kind, dtype, mode, B, Hq, Hkv, S, Dc, Dr, Dv, qk_norm=False, delta="shared", mask="causal"):
    c = dict(kind=kind, dtype=dtype, mode=mode, B=B, Hq=Hq, Hkv=Hkv, S=S, Dc=Dc, Dr=Dr, Dv=Dv, qk_norm=qk_norm,
             delta=delta if mode == "pope" else "none", mask=mask)
    return dict(name=name, **c) if name else c


def _decode(name, dtype, mode, B, Hq, Hkv, L, Sq, Dc, Dr, Dv, qk_norm=False):
    c = dict(kind="decode", dtype=dtype, mode=mode, B=B, Hq=Hq, Hkv=Hkv, L=L, Sq=Sq, Dc=Dc, Dr=Dr, Dv=Dv,
             qk_norm=qk_norm)
    return dict(name=name, **c) if name else c


def _block(name, pe_mode, B, S, hidden, Hq, Hkv):
    c = dict(kind="block", pe_mode=pe_mode, B=B, S=S, hidden=hidden, Hq=Hq, Hkv=Hkv)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # generation at the reference's model shape (content 64 + PoPE 2 x 32, 8 -> 4 heads): the next
        # token of one short sequence, the smallest call there is
        _decode("decode_short", "bf16", "pope", 1, 8, 4, 500, 1, 64, 32, 64),
        # the next token of one long sequence at the long-context attention shape (16 heads, fused PoPE)
        _decode("decode_long", "bf16", "pope", 1, 16, 16, 16384, 1, 0, 128, 128),
        # the next token of a batch of sequences, reference model shape
        _decode("decode_batch", "bf16", "pope", 16, 8, 4, 1999, 1, 64, 32, 64),
        # a prompt prefilled in pieces: 700 new rows behind 5300 cached ones
        _decode("prefill_chunk", "bf16", "pope", 1, 16, 16, 6000, 700, 0, 128, 128),
        # the reference trainer's attention step (B = 8, S = 512, 8 -> 4 heads, split form)
        _attn("split_train", "train", "bf16", "pope", 8, 8, 4, 512, 64, 32, 64),
        # the long-context training step, the package's headline
        _attn("pope_16k", "train", "bf16", "pope", 1, 16, 16, 16384, 0, 128, 128, delta="head"),
        # the RoPE + QKNorm arm at a common grouped-query shape (16 -> 4 heads of 128)
        _attn("rope_train", "train", "bf16", "rope", 4, 16, 4, 2048, 0, 128, 128, qk_norm=True),
        # fp16 mixed precision at the ~125M GPT shape (12 heads of 64), a length that fills no tile
        _attn("fp16_train", "train", "fp16", "pope", 8, 12, 12, 1000, 0, 64, 64, delta="head"),
        # padded batches: a key-padding mask and no causal mask
        _attn("masked_train", "train", "bf16", "pope", 2, 16, 16, 4096, 0, 128, 128, delta="head", mask="keypad"),
        # fp32 training of the reference's split form, 8 -> 4 heads
        _attn("train32", "train", "fp32", "pope", 4, 8, 4, 1024, 64, 32, 64),
        # the reference's 16k evaluation, which runs in fp32
        _attn("eval32", "eval", "fp32", "pope", 1, 16, 16, 16384, 0, 128, 128, delta="head"),
        # a whole transformer block of the reference's trainer: split PoPE with QK RMSNorm, hidden 512
        _block("block_train", "pope", 8, 512, 512, 8, 4),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm; odd ones among them."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _heads(rng, most):
    hkv = rng.choice([h for h in (1, 2, 3, 4, 6, 8, 12, 16) if h <= most])
    return hkv * rng.choice([g for g in (1, 1, 2, 4, 8) if hkv * g <= most]), hkv


def draw(rng):
    path = rng.choice(["decode", "decode", "chunk", "bf16", "bf16", "rope", "fp16", "masked", "train32", "eval32", "block"])
    if path in ("decode", "chunk"):
        mode = rng.choice(["pope", "pope", "split", "split", "rope"])
        hq, hkv = _heads(rng, 16)
        dc, dr, dv = {"pope": rng.choice([(0, 64, 64), (0, 128, 128)]), "split": (64, 32, 64),
                      "rope": rng.choice([(0, 64, 64), (0, 128, 128)])}[mode]
        if path == "decode":
            L, B, sq = _log(rng, 64, 16384), _log(rng, 1, 32), rng.choice([1, 1, 1, 1, 2, 4])
            B = max(1, min(B, 1 << 20 >> max(1, (L * hkv).bit_length() - 1)))
        else:
            L, B = _log(rng, 512, 12000), rng.choice([1, 1, 2])
            sq = min(L // 2, _log(rng, 32, 2048))
        return _decode(None, rng.choice(["bf16", "bf16", "bf16", "fp16"]), "rope" if mode == "rope" else "pope", B, hq,
                       hkv, L, sq, dc, dr, dv, qk_norm=mode == "rope" and rng.random() < 0.7)
    if path == "block":
        hidden, hq, hkv = rng.choice([(512, 8, 4), (512, 8, 8), (768, 12, 12), (768, 12, 4)])
        return _block(None, rng.choice(["pope", "pope", "rope"]), _log(rng, 1, 8), _log(rng, 100, 1024), hidden, hq, hkv)
    S = _log(rng, 100, 8192 if path in ("bf16", "eval32") else 4096)
    hq, hkv = _heads(rng, 16)
    most = {"train32": 3.0e8, "eval32": 1.5e9}.get(path, 2.0e9)  # query-key pairs
    hq, hkv = (hq, hkv) if hq * S * S <= most else (max(1, hq // hkv), 1)
    B = max(1, min(_log(rng, 1, 16), int(most / (hq * float(S) * S))))
    fused = rng.choice([(0, 64, 64), (0, 128, 128)])
    if path == "rope":
        return _attn(None, "train", rng.choice(["bf16", "bf16", "fp16"]), rng.choice(["rope", "rope", "none"]), B, hq, hkv, S,
                     *fused, qk_norm=rng.random() < 0.7)
    split = rng.random() < 0.5
    dims = (64, 32, 64) if split else fused
    delta = rng.choice(["shared", "head"])
    if path == "masked":
        return _attn(None, "train", rng.choice(["bf16", "bf16", "fp16"]), "pope", B, hq, hkv, S, *fused, delta=delta,
                     mask="keypad")
    kind, dtype = {"bf16": ("train", "bf16"), "fp16": ("train", "fp16"), "train32": ("train", "fp32"),
                   "eval32": ("eval", "fp32")}[path]
    return _attn(None, kind, dtype, "pope", B, hq, hkv, S, *dims, delta=delta)


# ------------------------------------------------------------------------------------------------ inputs

def _freqs(c):
    if c["mode"] == "pope":
        return 10000.0 ** (-(torch.arange(0, c["Dr"], dtype=torch.float32) / c["Dr"]))
    if c["mode"] == "rope":
        return 10000.0 ** (-(torch.arange(0, c["Dr"], 2, dtype=torch.float32) / c["Dr"]))
    return None


def _scale(c):
    """The split form and RoPE as their modules scale, the fused form 1/sqrt(D)."""
    return (c["Dc"] + 2 * c["Dr"]) ** -0.5 if c["Dc"] else c["Dr"] ** -0.5


def _inputs(c, seed, S, Sk):
    """The projections' (B, S, H * D) outputs viewed as (B, H, S, D), N(0, 1) as RMS-normed
    projections are; the phase bias U(-2 pi, 0)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPE[c["dtype"]]

    def proj(H, n, D):
        return torch.randn(c["B"], n, H, D, generator=g, device="cuda").to(dt).transpose(1, 2)

    x = {"q": proj(c["Hq"], S, c["Dr"]), "k": proj(c["Hkv"], Sk, c["Dr"]), "v": proj(c["Hkv"], Sk, c["Dv"])}
    if c["Dc"]:
        x["q_c"], x["k_c"] = proj(c["Hq"], S, c["Dc"]), proj(c["Hkv"], Sk, c["Dc"])
    if c["mode"] == "pope":
        shape = (c["Hkv"], c["Dr"]) if c.get("delta") == "head" else (c["Dr"],)
        x["delta"] = torch.rand(shape, generator=g, device="cuda") * (-2 * math.pi)
    return x, g


def _keep(c):
    """Keys that each batch entry keeps under the padding mask: all of them, then fewer and fewer."""
    return [c["S"] - (b * c["S"]) // (8 * c["B"]) for b in range(c["B"])]


def _mask(c):
    keep = torch.tensor(_keep(c), device="cuda").view(-1, 1)
    return (torch.arange(c["S"], device="cuda").view(1, -1) < keep).view(c["B"], 1, 1, c["S"])


def _block_module(c, seed):
    torch.manual_seed(seed)
    cfg = TransformerConfig(vocab_size=1024, hidden_dim=c["hidden"], num_layers=1, num_heads=c["Hq"], num_kv_heads=c["Hkv"],
                            head_dim=64, pe_mode=c["pe_mode"], max_seq_len=1024)
    pope = rope = None
    if c["pe_mode"] == "pope":
        pope = PoPEEmbedding(cfg.pope_d_rope, max_seq_len=1024, delta_init="uniform")
    else:
        rope = RotaryEmbedding(64, 1024)
    block = TransformerBlock(cfg, rope=rope, pope=pope).cuda()
    g = torch.Generator(device="cuda").manual_seed(seed + 1)
    with torch.no_grad():
        for name, p in block.named_parameters():
            if "norm" in name:
                p.copy_(1 + 0.05 * torch.randn(p.shape, generator=g, device="cuda"))
            elif p.dim() == 2:
                p.copy_(0.02 * torch.randn(p.shape, generator=g, device="cuda"))
    return block, g


def prepare(case, seed):
    c = case
    if c["kind"] == "block":
        block, g = _block_module(c, seed)
        x = torch.randn(c["B"], c["S"], c["hidden"], generator=g, device="cuda").requires_grad_()
        dy = torch.randn(c["B"], c["S"], c["hidden"], generator=g, device="cuda")
        return {"case": c, "block": block, "x": x, "dy": dy, "leaves": [x] + list(block.parameters())}
    freqs = _freqs(c)
    freqs = None if freqs is None else freqs.cuda()
    if c["kind"] == "decode":
        L, Sq, old = c["L"], c["Sq"], c["L"] - c["Sq"]
        x, _ = _inputs(c, seed, Sq, L)
        wk, wv = cache_widths(mode=c["mode"], d_content=c["Dc"], d_pe=c["Dr"], d_v=c["Dv"])
        cap = L + 64
        dt = DTYPE[c["dtype"]]
        kc = torch.zeros(c["B"], c["Hkv"], cap, wk, dtype=dt, device="cuda")
        vc = torch.zeros(c["B"], c["Hkv"], cap, wv, dtype=dt, device="cuda")
        kw = dict(mode=c["mode"], freqs=freqs, qk_norm=c["qk_norm"])
        cut = (lambda t, a, b: None if t is None else t[:, :, a:b])  # noqa: E731
        pe_cache_append(cut(x["k"], 0, old), cut(x["v"], 0, old), kc, vc, start_pos=0, k_c=cut(x.get("k_c"), 0, old),
                        delta=x.get("delta"), **kw)
        new = {n: cut(x.get(n), old, L) for n in ("k", "v", "k_c")}
        return {"case": c, "q": x["q"], "q_c": x.get("q_c"), "new": new, "delta": x.get("delta"), "kc": kc, "vc": vc,
                "kw": kw, "scale": _scale(c)}
    x, g = _inputs(c, seed, c["S"], c["S"])
    s = {"case": c, "x": x, "kw": dict(mode=c["mode"], freqs=freqs, scale=_scale(c), qk_norm=c["qk_norm"], causal=True)}
    if c["mask"] == "keypad":
        s["kw"].update(causal=False, mask=_mask(c))
    if c["kind"] == "train":
        for t in x.values():
            t.requires_grad_()
        s["dout"] = torch.randn(c["B"], c["S"], c["Hq"], c["Dv"], generator=g,
                                device="cuda").to(DTYPE[c["dtype"]]).transpose(1, 2)
    return s


# ------------------------------------------------------------------------------------------------ one pass

def run(state):
    c = state["case"]
    if c["kind"] == "block":
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = state["block"](state["x"])
        return [y.detach()] + list(torch.autograd.grad(y, state["leaves"], state["dy"]))
    if c["kind"] == "decode":
        new, L, old = state["new"], c["L"], c["L"] - c["Sq"]
        with torch.no_grad():
            pe_cache_append(new["k"], new["v"], state["kc"], state["vc"], start_pos=old, k_c=new["k_c"],
                            delta=state["delta"], **state["kw"])
            out, lse = pe_attention_decode(state["q"], state["kc"], state["vc"], L, d_v=c["Dv"], q_c=state["q_c"],
                                           scale=state["scale"], return_lse=True, **state["kw"])
        return {"out": out, "lse": lse, "k_rows": state["kc"][:, :, old:L], "v_rows": state["vc"][:, :, old:L]}
    x = state["x"]
    if c["kind"] == "eval":
        with torch.inference_mode():
            out, lse = pe_attention(**x, **state["kw"], return_lse=True)
        return {"out": out, "lse": lse}
    out = pe_attention(**x, **state["kw"])
    grads = torch.autograd.grad(out, list(x.values()), state["dout"])
    return {"out": out.detach(), **{"d" + n: g for n, g in zip(x, grads)}}


# ------------------------------------------------------------------------------------------------ bounds

def _widths(c):
    return c["Dc"] + (2 * c["Dr"] if c["mode"] == "pope" else c["Dr"]), c["Dv"]


def work(case):
    c = case
    if c["kind"] == "block":
        block = 64 + 2 * 32 if c["pe_mode"] == "pope" else 64
        h, tok = c["hidden"], c["B"] * c["S"]
        ffn = 256 * ((int(4 * h * 2 / 3) + 255) // 256)
        params = h * (c["Hq"] * (96 if c["pe_mode"] == "pope" else 64) + c["Hkv"] * (160 if c["pe_mode"] == "pope" else 128))
        params += h * c["Hq"] * 64 + 3 * h * ffn
        pairs = c["B"] * c["Hq"] * c["S"] ** 2 / 2
        return {"bytes": 4.0 * (4 * tok * h + 2 * params), "flops": 6.0 * params * tok + 2 * pairs * (4 * block + 3 * 64)}
    e = 4 if c["dtype"] == "fp32" else 2
    wqk, dv = _widths(c)
    raw = c["Dc"] + c["Dr"]
    if c["kind"] == "decode":
        n = c["Sq"]
        pairs = c["B"] * c["Hq"] * (n * (c["L"] - n) + n * (n + 1) / 2)
        rows = c["B"] * c["Hkv"]
        return {"bytes": e * float(rows * c["L"] * (wqk + dv) + rows * n * (raw + dv + wqk + dv) + c["B"] * c["Hq"] * n * (raw + dv)),
                "flops": 2.0 * pairs * (wqk + dv)}
    pairs = c["B"] * c["Hq"] * (c["S"] ** 2 / 2.0) if c["mask"] == "causal" else c["Hq"] * c["S"] * float(sum(_keep(c)))
    q, kv = c["B"] * c["Hq"] * c["S"], c["B"] * c["Hkv"] * c["S"]
    io = q * (raw + dv) + kv * (raw + dv)  # q, out and k, v
    if c["kind"] == "eval":
        return {"bytes": float(e * io), "flops": 2.0 * pairs * (wqk + dv)}
    return {"bytes": float(e * (2 * io)), "flops": 2.0 * pairs * (4 * wqk + 3 * dv)}


def tolerance(case):
    """About four times the largest error against ``exact`` that was measured over the listed and some
    drawn cases: in bf16 0.0028 (forward, decode), 0.006 (gradients; the shared phase bias's) and
    0.0074 (a block's parameter gradients), in fp16 0.0006, in fp32 7.7e-7."""
    c = case
    if c["kind"] == "block":
        return {"rel": 0.03}
    if c["dtype"] == "fp32":
        return {"rel": 4e-6}
    if c["dtype"] == "fp16":
        return {"rel": 0.0025}
    return {"rel": 0.02 if c["kind"] == "train" else 0.012}


# ------------------------------------------------------------------------------------------------ the same in 64 bits

def _angles(n, freqs, start):
    """The phases as the reference forms them: one fp32 product of position and frequency."""
    return torch.arange(start, start + n, dtype=torch.float32, device="cuda").view(-1, 1) * freqs.cuda().view(1, -1)


def _transform(x, mode, freqs, start, delta=None):
    """(B, H, S, D) in 64 bits -> PoPE's [mu cos, mu sin] or the rotated pairs."""
    if mode == "none":
        return x
    ph = _angles(x.shape[2], freqs, start)
    if mode == "pope":
        mu = F.softplus(x)
        if delta is None:
            ph = ph.double()
        else:  # (D,) or (H, D): the fp32 sum, with the derivative of the sum
            d = delta.view(1, 1, 1, -1) if delta.dim() == 1 else delta.view(1, delta.shape[0], 1, -1)
            ph = (ph + d.detach().float()).double() + (d - d.detach())
        return torch.cat([mu * ph.cos(), mu * ph.sin()], -1)
    c, s = ph.double().cos(), ph.double().sin()
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack([x0 * c - x1 * s, x0 * s + x1 * c], -1).flatten(-2)


def _operands(c, x, start_q):
    qt = _transform(x["q"], c["mode"], _freqs(c), start_q)
    kt = _transform(x["k"], c["mode"], _freqs(c), 0, x.get("delta"))
    if c["qk_norm"]:
        qt, kt = (t / (t.norm(dim=-1, keepdim=True) + 1e-6) for t in (qt, kt))
    if c["Dc"]:
        qt, kt = torch.cat([x["q_c"], qt], -1), torch.cat([x["k_c"], kt], -1)
    return qt, kt


def _visible(c, b, sq, sk):
    if c.get("mask") == "keypad":
        return (torch.arange(sk, device="cuda") < _keep(c)[b]).view(1, -1).expand(sq, sk)
    i = torch.arange(sq, device="cuda").view(-1, 1) + (sk - sq)
    return torch.arange(sk, device="cuda").view(1, -1) <= i


def _attention64(c, qt, kt, v, dout=None):
    """softmax(scale q k^T) v head by head in 64 bits, and the gradients of qt, kt and v in closed form."""
    B, H, Sq, _ = qt.shape
    grp, scale = H // kt.shape[1], _scale(c)
    out = torch.empty(B, H, Sq, v.shape[-1], dtype=torch.float64, device="cuda")
    lse = torch.empty(B, H, Sq, dtype=torch.float64, device="cuda")
    dq, dk, dv = (torch.zeros_like(t) for t in (qt, kt, v)) if dout is not None else (None, None, None)
    for b in range(B):
        see = _visible(c, b, Sq, kt.shape[2])
        for h in range(H):
            q, k, w = qt[b, h], kt[b, h // grp], v[b, h // grp]
            s = (q @ k.T).mul_(scale).masked_fill_(~see, -math.inf)
            lse[b, h] = torch.logsumexp(s, -1)
            p = s.sub_(lse[b, h].unsqueeze(-1)).exp_()
            out[b, h] = p @ w
            if dout is not None:
                do = dout[b, h]
                dv[b, h // grp] += p.T @ do
                ds = (do @ w.T).sub_((do * out[b, h]).sum(-1, keepdim=True)).mul_(p).mul_(scale)
                dq[b, h] = ds @ k
                dk[b, h // grp] += ds.T @ q
    return out, lse, dq, dk, dv


def _block64(c, block, x):
    P = {n: p.detach().double().requires_grad_() for n, p in block.named_parameters()}
    B, S, Hq, Hkv = c["B"], c["S"], c["Hq"], c["Hkv"]

    def norm(t, w):
        return t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + 1e-6) * w

    def heads(t, H):
        return t.view(B, S, H, -1).transpose(1, 2)

    h = norm(x, P["attention_norm.weight"])
    a = "attention."
    if c["pe_mode"] == "pope":
        f = 10000.0 ** (-(torch.arange(0, 32, dtype=torch.float32) / 32))
        qr = norm(h @ P[a + "wq_r.weight"].T, P[a + "qr_norm.weight"])
        kr = norm(h @ P[a + "wk_r.weight"].T, P[a + "kr_norm.weight"])
        delta = P[a + "fpope.phase_bias"].clamp(-2 * math.pi, 0.0)
        q = torch.cat([heads(h @ P[a + "wq_c.weight"].T, Hq), _transform(heads(qr, Hq), "pope", f, 0)], -1)
        k = torch.cat([heads(h @ P[a + "wk_c.weight"].T, Hkv), _transform(heads(kr, Hkv), "pope", f, 0, delta)], -1)
    else:
        f = 10000.0 ** (-(torch.arange(0, 64, 2, dtype=torch.float32) / 64))
        q, k = (_transform(heads(h @ P[a + n + ".weight"].T, H), "rope", f, 0) for n, H in (("wq", Hq), ("wk", Hkv)))
        q, k = (t / (t.norm(dim=-1, keepdim=True) + 1e-6) for t in (q, k))
    v = heads(h @ P[a + "wv.weight"].T, Hkv)
    k, v = (t.repeat_interleave(Hq // Hkv, 1) for t in (k, v))
    s = (q @ k.transpose(-1, -2)) * q.shape[-1] ** -0.5
    s = s.masked_fill(torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1), -math.inf)
    o = (s.softmax(-1) @ v).transpose(1, 2).reshape(B, S, -1)
    y = x + o @ P[a + "wo.weight"].T
    h = norm(y, P["ffn_norm.weight"])
    g = F.silu(h @ P["feed_forward.w3.weight"].T) * (h @ P["feed_forward.w1.weight"].T)
    return y + g @ P["feed_forward.w2.weight"].T, list(P.values())


def exact(case, seed):
    c = case
    if c["kind"] == "block":
        st = prepare(c, seed)
        x = st["x"].detach().double().requires_grad_()
        y, params = _block64(c, st["block"], x)
        return [y.detach()] + list(torch.autograd.grad(y, [x] + params, st["dy"].double()))
    if c["kind"] == "decode":
        x, _ = _inputs(c, seed, c["Sq"], c["L"])
        x = {n: t.double() for n, t in x.items()}
        qt, kt = _operands(c, x, c["L"] - c["Sq"])
        out, lse, *_ = _attention64(c, qt, kt, x["v"])
        old, (wk, wv) = c["L"] - c["Sq"], cache_widths(mode=c["mode"], d_content=c["Dc"], d_pe=c["Dr"], d_v=c["Dv"])
        return {"out": out, "lse": lse, "k_rows": F.pad(kt[:, :, old:], (0, wk - kt.shape[-1])),
                "v_rows": F.pad(x["v"][:, :, old:], (0, wv - c["Dv"]))}
    x, g = _inputs(c, seed, c["S"], c["S"])
    train = c["kind"] == "train"
    x = {n: t.double().requires_grad_(train) for n, t in x.items()}
    qt, kt = _operands(c, x, 0)
    if not train:
        out, lse, *_ = _attention64(c, qt, kt, x["v"])
        return {"out": out, "lse": lse}
    dout = torch.randn(c["B"], c["S"], c["Hq"], c["Dv"], generator=g, device="cuda").to(DTYPE[c["dtype"]])
    with torch.no_grad():
        out, _, dq, dk, dv = _attention64(c, qt, kt, x["v"], dout.transpose(1, 2).double())
    names = [n for n in x if n != "v"]
    grads = dict(zip(names, torch.autograd.grad([qt, kt], [x[n] for n in names], [dq, dk])), v=dv)
    return {"out": out, **{"d" + n: grads[n] for n in x}}
