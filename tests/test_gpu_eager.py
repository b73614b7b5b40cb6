"""The eager differentiable paths that pass the operators by: the operators' outputs and gradients
(bit for bit but where a residual sum is not used), and the operators themselves wherever something
watches the call."""
from __future__ import annotations

import pytest
import torch

import fused_layernorm as fl
from fused_layernorm import ops as fops

pytestmark = pytest.mark.gpu

DEV = "cuda"
KINDS = ["ln", "rms", "gelu_tanh", "gelu_none", "add_ln", "add_rms"]


def _call(kind, x, r, shape, w, b):
    if kind == "ln":
        return (fl.fused_layer_norm(x, shape, w, b, 1e-5),)
    if kind == "rms":
        return (fl.fused_rms_norm(x, shape, w, 1e-5),)
    if kind.startswith("gelu"):
        return (fops.layer_norm_gelu(x, shape, w, b, 1e-5, approximate=kind[5:]),)
    if kind == "add_ln":
        return fops.add_layer_norm(x, r, shape, w, b, 1e-5)
    return fops.add_rms_norm(x, r, shape, w, 1e-5)


def _inputs(kind, dtype, lead, shape, affine=True, strided=False):
    g = torch.Generator().manual_seed(7)

    def leaf(*s):
        t = torch.randn(*s, generator=g).to(DEV, dtype)
        if strided:
            t = t.transpose(0, 1).contiguous().transpose(0, 1)
        return t.requires_grad_()

    x = leaf(*lead, *shape)
    r = leaf(*lead, *shape) if kind.startswith("add") else None
    w = b = None
    if affine:
        w = torch.randn(*shape, generator=g).to(DEV, dtype).requires_grad_()
        b = torch.randn(*shape, generator=g).to(DEV, dtype).requires_grad_()
    if "rms" in kind:
        b = None
    return x, r, w, b


def _step(kind, x, r, shape, w, b, use=(True, True)):
    out = _call(kind, x, r, shape, w, b)
    g = torch.Generator().manual_seed(11)
    ups = [torch.randn(*o.shape, generator=g).to(o) for o in out]
    picked = [(o, u) for o, u, k in zip(out, ups, use) if k]
    leaves = [t for t in (x, r, w, b) if t is not None]
    grads = torch.autograd.grad([o for o, _ in picked], leaves, [u for _, u in picked],
                                allow_unused=True)
    return [o.detach() for o in out], grads


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("dtype,lead,shape,affine,strided", [
    (torch.bfloat16, (5, 7), (4, 6, 33), True, False), (torch.float32, (), (2, 129), True, False),
    (torch.float16, (40,), (768,), False, False), (torch.float32, (6, 9), (3, 64), True, True)])
def test_eager_paths_equal_the_operators(monkeypatch, kind, dtype, lead, shape, affine, strided):
    for use in ((True, True), (True, False), (False, True)):
        if use != (True, True) and not kind.startswith("add"):
            continue
        args = _inputs(kind, dtype, lead, shape, affine, strided)
        x, r, w, b = args
        got = _step(kind, x, r, shape, w, b, use)
        with monkeypatch.context() as m:
            m.setattr(fops, "_ordinary", lambda *t: False)
            want = _step(kind, x, r, shape, w, b, use)
        for a, c in zip(got[0] + list(got[1]), want[0] + list(want[1])):
            assert (a is None) == (c is None)
            if a is None or (a.shape == c.shape and torch.equal(a, c)):
                continue
            # The operators fill in zeros for the gradient of an unused h and add them in the
            # kernel's residual form, which rounds the sum to fp32 before the output type; without
            # them the last FMA rounds to the output type directly.  Both are within half an ulp
            # plus half an fp32 ulp of the same value, so at most one ulp apart.
            assert use == (True, False) and a.shape == c.shape, kind
            ulp = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
            err = (a.float() - c.float()).abs()
            assert (err <= ulp * c.float().abs() + 2.0 ** -24).all() and dtype != torch.float32


@pytest.mark.parametrize("kind", ["gelu_tanh", "add_rms"])
def test_watched_calls_take_the_operators(kind):
    """Dispatch modes see the operators, tangents and functorch transforms meet their rules, saved
    tensor hooks see what is saved, and in-place changes of it are caught."""
    from torch.utils._python_dispatch import TorchDispatchMode
    shape = (4, 64)
    x, r, w, b = _inputs(kind, torch.float32, (6,), shape)
    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Watch():
        out = _call(kind, x, r, shape, w, b)
        torch.autograd.grad(out[0].sum(), x)
    assert any("_fwd" in f for f in seen) and any("_bwd" in f for f in seen), seen
    out = _call(kind, x, r, shape, w, b)
    seen.clear()
    with Watch():  # the forward ran unwatched, its backward does not
        torch.autograd.grad(out[0].sum(), x)
    assert any("fused_layernorm" in f and "_bwd" in f for f in seen), seen
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x.detach(), torch.ones_like(x))
        with pytest.raises(NotImplementedError):
            _call(kind, dual, r, shape, w, b)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t,
                                                  lambda t: t):
        out = _call(kind, x, r, shape, w, b)
    assert len(packed) >= 3
    torch.autograd.grad(out[0].sum(), x)
    y = _call(kind, x.clone(), r, shape, w, b)[0]
    with torch.no_grad():
        w.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()


def test_parameters_that_were_refused_stay_refused():
    x = torch.randn(4, 64, device=DEV)
    for w in (torch.ones(128, device=DEV)[::2], torch.ones(32, device=DEV),
              torch.ones(64, device=DEV, dtype=torch.float16), torch.ones(64)):
        with pytest.raises(RuntimeError):
            fops.add_rms_norm(x, x, 64, w)
        with pytest.raises(RuntimeError):
            fops.layer_norm_gelu(x, (64,), w, None)
    with pytest.raises(RuntimeError):
        fops.layer_norm_gelu(x, (32,), None, None)
    with pytest.raises(RuntimeError):
        fops.layer_norm_gelu(x, (64,), None, None, approximate="erf")


def test_quantized_forwards_pass_gradients_through_h():
    x, r, w, _ = _inputs("add_rms", torch.bfloat16, (6,), (64,))
    q, s, h = fops.add_rms_norm_mxfp8(x, r, 64, w)
    torch.testing.assert_close(torch.autograd.grad(h.sum(), x)[0], torch.ones_like(x))
    with torch.no_grad():
        q2, s2, h2 = fops.add_rms_norm_mxfp8(x, r, 64, w)
    assert torch.equal(q.view(torch.uint8), q2.view(torch.uint8)) and torch.equal(h, h2)
    assert torch.equal(s.view(torch.uint8), s2.view(torch.uint8)) and not h2.requires_grad


@pytest.mark.parametrize("kind,lead,shape", [(k, (5, 3), (4, 33)) for k in KINDS]
                         + [("ln", (5, 3), (132,)), ("rms", (15,), (132,)),
                            ("add_rms", (15,), (132,)), ("gelu_tanh", (132,), (132,))])
@pytest.mark.parametrize("affine", [True, False])
@pytest.mark.parametrize("backend", ["eager", "aot_eager"])
def test_backward_under_compiled_autograd(kind, lead, shape, affine, backend):
    """A forward in eager code whose backward compiled autograd captures: the eager gradients."""
    from torch._dynamo import compiled_autograd
    torch._dynamo.reset()
    for use in ((True, True), (True, False), (False, True))[:3 if kind.startswith("add") else 1]:
        x, r, w, b = _inputs(kind, torch.float32, lead, shape, affine)
        _, want = _step(kind, x, r, shape, w, b, use)
        out = _call(kind, x, r, shape, w, b)
        g = torch.Generator().manual_seed(11)
        ups = [torch.randn(*o.shape, generator=g).to(o) for o in out]
        loss = sum((o * u).sum() for o, u, k in zip(out, ups, use) if k)
        with compiled_autograd._enable(torch.compile(backend=backend, fullgraph=True)):
            loss.backward()
        for t, c in zip([t for t in (x, r, w, b) if t is not None], want):
            # (a gradient that reaches nothing is zeros in one and absent in the other)
            got = torch.zeros_like(t) if t.grad is None else t.grad
            assert torch.equal(got, torch.zeros_like(t) if c is None else c)


def test_zero_tensors_stay_refused():
    """torch's tensors of zeros without storage: the operators refuse what their dispatch makes of
    them (an expanded zero); a null gamma would be taken for an absent one."""
    x = torch.randn(6, 64, device=DEV)
    zero, big = (torch._efficientzerotensor(s, device=DEV) for s in ((64,), (6, 64)))
    y = fops.layer_norm_gelu(x.clone().requires_grad_(), 64)
    for call in (lambda: fops.add_rms_norm(x, x, 64, zero),
                 lambda: fops.layer_norm_gelu(x, 64, zero, zero),
                 lambda: fops.rms_norm_fp8(x, 64, zero), lambda: fops.add_layer_norm(x, big, 64),
                 lambda: y.backward(big)):
        with pytest.raises(RuntimeError, match="must be contiguous"):
            call()
