"""RMSNorm and SwiGLU in training: the modules' fused Functions against the torch expressions they stand for.

Rows of one to 8192 features in every dtype pair the module sends to the kernel, non-contiguous inputs,
single gradients, second derivatives, and the callers that must see the torch ops (vmap, forward mode,
functorch grad, a dispatch mode), which take the expression.  Tolerances: fp32 sums in another order, 2e-6
relative to the largest entry (dw sums over the rows: times sqrt(rows) / 8); bf16 results one rounding,
2^-7 of the largest entry.
"""

import pytest
import torch
import torch.nn.functional as F

from pe_ablations_amd.ffn import SwiGLU
from pe_ablations_amd.functional import rms_norm_expression
from pe_ablations_amd.normalization import RMSNorm

pytestmark = pytest.mark.gpu
F32, B16 = torch.float32, torch.bfloat16


def near(a, b, tol):
    return (a.double() - b.double()).abs().max() <= tol * b.double().abs().max().clamp_min(1e-30)


@pytest.mark.parametrize("shape,xt,wt", [((1, 8), F32, F32), ((3, 5, 512), F32, F32), ((2, 70, 768), B16, F32),
                                         ((129, 2048), B16, B16), ((7, 8192), F32, F32), ((2, 33, 520), F32, B16)])
def test_rmsnorm_gradients(cuda, shape, xt, wt):
    g = torch.Generator(device="cuda").manual_seed(shape[-1])
    m = RMSNorm(shape[-1]).cuda()
    m.weight.data = (1 + 0.1 * torch.randn(shape[-1], generator=g, device="cuda")).to(wt)
    x = torch.randn(shape, generator=g, device="cuda").to(xt).requires_grad_()
    y = m(x)
    ref = rms_norm_expression(x, m.weight, m.eps)
    assert y.grad_fn.name().startswith("RMSNormFn") and y.dtype == ref.dtype
    dy = torch.randn(y.shape, generator=g, device="cuda").to(y.dtype)
    rows = x.numel() // shape[-1]
    got, want = torch.autograd.grad(y, (x, m.weight), dy), torch.autograd.grad(ref, (x, m.weight), dy)
    half = (lambda t: 2 ** -7 if t.dtype == B16 else 2e-6)  # noqa: E731
    assert near(y, ref, half(ref))
    # with any 16-bit tensor in the chain, an intermediate may round the other way in either result
    assert near(got[0], want[0], 2 ** -7 if B16 in (xt, wt) else 2e-6)
    assert near(got[1], want[1], 2 ** -7 if B16 in (xt, wt) else 2e-6 * max(1.0, rows ** 0.5 / 8))


def test_rmsnorm_views_and_single_gradients(cuda):
    m = RMSNorm(64).cuda()
    base = torch.randn(64, 40, device="cuda", requires_grad=True)
    y = m(base.t())
    ref = rms_norm_expression(base.t(), m.weight, m.eps)
    dy = torch.randn(64, 40, device="cuda").t()
    assert near(torch.autograd.grad(y, base, dy)[0], torch.autograd.grad(ref, base, dy)[0], 2e-6)
    x = torch.randn(5, 64, device="cuda")
    y, ref = m(x), rms_norm_expression(x, m.weight, m.eps)  # the weight alone
    assert near(torch.autograd.grad(y.sum(), m.weight)[0], torch.autograd.grad(ref.sum(), m.weight)[0], 2e-6)
    m.weight.requires_grad_(False)
    x.requires_grad_()
    # the input alone (cubes: a row's squares sum to a constant, whose gradient is rounding noise only); y^2
    # and the sums round a few times more than y: 4e-6
    y, ref = m(x), rms_norm_expression(x, m.weight, m.eps)
    assert near(torch.autograd.grad(y.pow(3).sum(), x)[0], torch.autograd.grad(ref.pow(3).sum(), x)[0], 4e-6)


def test_second_derivatives(cuda):
    m = RMSNorm(32).cuda()
    x = torch.randn(6, 32, device="cuda", requires_grad=True)

    def second(y):
        g, = torch.autograd.grad(y.pow(3).sum(), x, create_graph=True)
        return torch.autograd.grad(g.square().sum(), (x, m.weight))

    for a, b in zip(second(m(x)), second(rms_norm_expression(x, m.weight, m.eps))):
        assert near(a, b, 1e-5)
    u, v = (torch.randn(4, 16, device="cuda").to(B16).requires_grad_() for _ in range(2))
    g, = torch.autograd.grad(SwiGLU()(u, v).float().square().sum(), v, create_graph=True)
    r, = torch.autograd.grad((F.silu(v) * u).float().square().sum(), v, create_graph=True)
    assert torch.equal(torch.autograd.grad(g.float().sum(), u)[0], torch.autograd.grad(r.float().sum(), u)[0])


def test_transforms_take_the_expression(cuda):
    m = RMSNorm(16).cuda()
    x, t = torch.randn(3, 5, 16, device="cuda"), torch.randn(3, 5, 16, device="cuda")
    ref = rms_norm_expression(x, m.weight, m.eps)
    assert near(torch.vmap(m)(x), ref, 2e-6)
    out, tangent = torch.func.jvp(lambda z: rms_norm_expression(z, m.weight, m.eps), (x,), (t,))
    out2, tangent2 = torch.func.jvp(m, (x,), (t,))
    assert near(tangent2, tangent, 2e-6) and near(out2, out, 2e-6)
    gf = torch.func.grad(lambda z: m(z).pow(3).sum())(x)
    assert near(gf, torch.func.grad(lambda z: rms_norm_expression(z, m.weight, m.eps).pow(3).sum())(x), 4e-6)
    with torch.autograd.forward_ad.dual_level():
        d = torch.autograd.forward_ad.make_dual(x, t)
        assert near(torch.autograd.forward_ad.unpack_dual(m(d)).tangent, tangent, 2e-6)
    from torch.fx.experimental.proxy_tensor import make_fx
    traced = make_fx(lambda z: m(z))(x.requires_grad_())
    assert any("rsqrt" in str(n.target) for n in traced.graph.nodes)


@pytest.mark.parametrize("shape", [(1, 8), (3, 1000), (2, 5, 1536)])
def test_swiglu_gradients(cuda, shape):
    g = torch.Generator(device="cuda").manual_seed(1)
    x, gate, dy = ((3 * torch.randn(shape, generator=g, device="cuda")).to(B16) for _ in range(3))
    x.requires_grad_(), gate.requires_grad_()
    y = SwiGLU()(x, gate)
    assert y.grad_fn.name().startswith("SwiGLUFn")
    ref = F.silu(gate) * x
    assert torch.equal(y, ref)
    got, want = torch.autograd.grad(y, (x, gate), dy), torch.autograd.grad(ref, (x, gate), dy)
    assert torch.equal(got[0], want[0])
    assert (got[1].float() - want[1].float()).abs().max() <= 2 ** -7 * want[1].float().abs().max()
    t = gate.detach().t().contiguous().t().requires_grad_() if gate.dim() == 2 else gate.detach().requires_grad_()
    assert torch.equal(torch.autograd.grad(SwiGLU()(x, t), t, dy)[0], got[1])  # a transposed gate


@pytest.mark.parametrize("xt", [F32, B16])
@pytest.mark.parametrize("what", ["x", "weight", "dy"])
def test_rmsnorm_unaligned_operands(cuda, xt, what):
    """Views two or four bytes past a 16-byte boundary: x and the weight take the expression, dy a copy."""
    def off(t, shift):
        flat = torch.empty(t.numel() + 8, dtype=t.dtype, device="cuda")
        v = flat[shift:shift + t.numel()].view(t.shape)
        v.copy_(t)
        return v.detach()
    g = torch.Generator(device="cuda").manual_seed(3)
    m = RMSNorm(64).cuda()
    m.weight.data = off(1 + 0.1 * torch.randn(64, generator=g, device="cuda"), int(what == "weight"))
    x = off(torch.randn(9, 64, generator=g, device="cuda").to(xt), int(what == "x")).requires_grad_()
    y, ref = m(x), rms_norm_expression(x, m.weight, m.eps)
    dy = off(torch.randn(9, 64, generator=g, device="cuda").to(y.dtype), int(what == "dy"))
    for a, b in zip(torch.autograd.grad(y, (x, m.weight), dy), torch.autograd.grad(ref, (x, m.weight), dy)):
        assert near(a, b, 2 ** -7 if xt == B16 else 2e-6)


def test_rmsnorm_half_input_changed_in_place_afterwards(cuda):
    m = RMSNorm(64).cuda()
    grads = []
    for norm in (m, lambda t: rms_norm_expression(t, m.weight, m.eps)):
        leaf = torch.linspace(-2, 3, 9 * 64, device="cuda").view(9, 64).to(B16).requires_grad_()
        x = leaf * 1.0
        y = norm(x)
        x += 1.0
        grads.append(torch.autograd.grad((y * y * y).sum() + x.sum(), leaf)[0])
    assert near(grads[0], grads[1], 2 ** -7)


def outcome(fn, make, needs, touch):
    """What a call and its backward give when the tensor named by ``touch`` is changed in place between the
    two: the gradients, or "error"."""
    t = make()
    for n in needs:
        t[n].requires_grad_()
    y = fn(t)
    if touch:
        with torch.no_grad():
            t[touch].add_(1.0)
    try:
        return torch.autograd.grad(y.sum(), [t[n] for n in needs])
    except RuntimeError:
        return "error"


@pytest.mark.parametrize("touch", ["", "x", "w"])
@pytest.mark.parametrize("needs", [("x",), ("w",), ("x", "w")])
@pytest.mark.parametrize("op", ["norm32", "norm16", "swiglu"])
def test_changes_in_place_are_refused_where_the_expression_refuses_them(cuda, op, needs, touch):
    def make():
        g = torch.Generator(device="cuda").manual_seed(11)
        x = torch.randn(6, 64, generator=g, device="cuda")
        w = torch.randn(6, 64, generator=g, device="cuda") if op == "swiglu" else 1 + 0.1 * torch.randn(64, generator=g, device="cuda")
        return {"x": x if op == "norm32" else x.to(B16), "w": w.to(B16) if op == "swiglu" else w}

    def module(t):
        if op == "swiglu":
            return SwiGLU()(t["x"], t["w"])
        m = RMSNorm(64).cuda()
        del m.weight
        m.weight = t["w"]
        return m(t["x"])

    def expression(t):
        return F.silu(t["w"]) * t["x"] if op == "swiglu" else rms_norm_expression(t["x"], t["w"], 1e-6)

    got, want = outcome(module, make, needs, touch), outcome(expression, make, needs, touch)
    assert (got == "error") == (want == "error")
    if got != "error":
        for a, b in zip(got, want):
            assert near(a, b, 2e-6 if op == "norm32" else 2 ** -7)


def test_inference_tensors_without_a_gradient(cuda):
    """Frozen features made under inference mode, in front of a norm that is trained."""
    with torch.inference_mode():
        x = torch.randn(6, 64, device="cuda")
    m = RMSNorm(64).cuda()
    dy = torch.randn(6, 64, device="cuda")
    got, = torch.autograd.grad(m(x), m.weight, dy)
    want, = torch.autograd.grad(rms_norm_expression(x.clone(), m.weight, m.eps), m.weight, dy)
    assert near(got, want, 2e-6)


def test_batched_gradients(cuda):
    """is_grads_batched and jacobian(vectorize=True), whose backward sees functorch tensors."""
    g = torch.Generator(device="cuda").manual_seed(13)
    m = RMSNorm(16).cuda()
    x = torch.randn(4, 16, generator=g, device="cuda", requires_grad=True)
    dys = torch.randn(5, 4, 16, generator=g, device="cuda")
    y, ref = m(x), rms_norm_expression(x, m.weight, m.eps)
    assert y.grad_fn.name().startswith("RMSNormFn")
    for a, b in zip(torch.autograd.grad(y, (x, m.weight), dys, is_grads_batched=True),
                    torch.autograd.grad(ref, (x, m.weight), dys, is_grads_batched=True)):
        assert near(a, b, 2e-6)
    jac = torch.autograd.functional.jacobian
    assert near(jac(m, x, vectorize=True), jac(lambda z: rms_norm_expression(z, m.weight, m.eps), x, vectorize=True), 2e-6)
    u, v, d = (torch.randn(n, 4, 16, generator=g, device="cuda").to(B16) for n in (1, 1, 5))
    u, v = u[0].requires_grad_(), v[0].requires_grad_()
    for a, b in zip(torch.autograd.grad(SwiGLU()(u, v), (u, v), d, is_grads_batched=True),
                    torch.autograd.grad(F.silu(v) * u, (u, v), d, is_grads_batched=True)):
        assert torch.equal(a, b)
