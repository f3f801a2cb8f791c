"""The fused inference layers call a projection that something stands around (a hook, an adapter, a replaced forward) at every
row count: with one that doubles its result, the layer's output is what the torch path gives. Tolerance (2-norm relative):
each projection, the layer's inner results and its output are rounded to bf16 (2^-9 in the mean) on either path, at most ~12 roundings a
path: 24 of them in quadrature 1e-2; fp32 sums of at most 1024 products and 12 levels 2e-5."""

import pytest
import torch
import torch.nn as nn

pytestmark = pytest.mark.gpu
DEV = "cuda"


class Doubled(nn.Linear):
    def forward(self, h):
        return 2 * super().forward(h)


def _around(l, kind):
    if kind == "hook":
        l.register_forward_hook(lambda m, i, o: 2 * o)
    elif kind == "replaced":
        l.forward = lambda h: 2 * nn.Linear.forward(l, h)
    else:
        ad = Doubled(l.in_features, l.out_features, bias=False).to(l.weight)
        ad.weight = l.weight
        return ad
    return l


def _layer(cls, dtype, d=256):
    import dispatcher_hybrid.modeling_dispatcher as md
    from dispatcher_hybrid import DispatcherConfig
    torch.manual_seed(11)
    layer = getattr(md, cls)(DispatcherConfig(d_model=d, num_heads=d // 64, max_len=4096, attn_window=128, num_layers=1,
                                              vocab_size=64, dim_feedforward=2 * d)).to(DEV, dtype)
    with torch.no_grad():
        for n, p in layer.named_parameters():
            if "bias" not in n:
                p.normal_(std=0.05)
    return layer.eval()


CASES = [  # layer, projection, dtype, b, T: whole-layer call, one launch, and the ranges where only some products are
    ("DispatcherMixer", "linear_out", torch.bfloat16, 1, 200), ("DispatcherMixer", "linear_out", torch.bfloat16, 1, 3000),
    ("DispatcherMixer", "gate_hidden", torch.bfloat16, 2, 3000), ("DispatcherMixer", "linear_out", torch.float32, 2, 1400),
    ("WindowAttention", "linear_q", torch.bfloat16, 2, 3000), ("WindowAttention", "linear_out", torch.bfloat16, 1, 3000),
    ("WindowAttention", "linear_v", torch.bfloat16, 1, 100), ("SwiGLU", "linear_gate", torch.bfloat16, 1, 100),
    ("SwiGLU", "linear_down", torch.bfloat16, 1, 100), ("SwiGLU", "linear_up", torch.float32, 1, 100)]


@pytest.mark.parametrize("kind", ["hook", "replaced", "adapter"])
@pytest.mark.parametrize("cls,proj,dtype,b,T", CASES)
def test_inference_calls_what_stands_around_a_projection(cls, proj, dtype, b, T, kind):
    layer = _layer(cls, dtype)
    setattr(layer, proj, _around(getattr(layer, proj), kind))
    x = torch.randn(b, T, 256, device=DEV).to(dtype)
    t = torch.arange(T, device=DEV).unsqueeze(1)
    args = (x, (t >= (1 << torch.arange(12, device=DEV))).to(dtype)) if cls == "DispatcherMixer" else (x,)
    with torch.no_grad():
        want = layer(*args)
        layer.use_fused_gates = layer.use_fused = True
        got = layer(*args)
    assert (got.double() - want.double()).norm() <= (1e-2 if dtype == torch.bfloat16 else 2e-5) * want.double().norm()


def test_a_hook_keeps_the_gate_it_was_given():
    layer = _layer("SwiGLU", torch.bfloat16)
    kept = []
    layer.linear_gate.register_forward_hook(lambda m, i, o: kept.append((o, o.clone())) and None)
    layer.use_fused = True
    with torch.no_grad():
        layer(torch.randn(1, 70, 256, device=DEV).bfloat16())
    assert torch.equal(*kept[0])


def _inputs(layer, cls, x):
    if cls != "DispatcherMixer":
        return (x,)
    t = torch.arange(x.shape[1], device=DEV).unsqueeze(1)
    return x, (t >= (1 << torch.arange(12, device=DEV))).to(x.dtype)


@pytest.mark.parametrize("cls,dtype", [("DispatcherMixer", torch.bfloat16), ("DispatcherMixer", torch.float32),
                                       ("WindowAttention", torch.bfloat16)])
def test_broadcast_gradients_and_inputs_in_training(cls, dtype):
    """A gradient or an input whose rows are one row in memory gives what its dense copy gives, bit for bit."""
    layer = _layer(cls, dtype)
    layer.use_fused_gates = layer.use_fused = True
    w = torch.randn(256, device=DEV).to(dtype)

    def grads(x, dy):
        x = x.detach().requires_grad_()
        layer.zero_grad()
        layer(*_inputs(layer, cls, x)).backward(dy)
        return [x.grad, *[p.grad for p in layer.parameters()]]

    x = torch.randn(2, 70, 256, device=DEV).to(dtype)
    for dy in (w.expand(2, 70, 256), torch.randn(2, 1, 256, device=DEV).to(dtype).expand(2, 70, 256)):
        for a, e in zip(grads(x, dy), grads(x, dy.contiguous())):
            assert torch.equal(a, e)
    row = w.clone().requires_grad_()
    y = layer(*_inputs(layer, cls, row.expand(2, 70, 256)))
    y.sum((0, 1)).square().sum().backward()
    assert torch.equal(y.detach(), layer(*_inputs(layer, cls, row.detach().expand(2, 70, 256).contiguous())).detach())
    assert row.grad.isfinite().all()


@pytest.mark.parametrize("cls,T", [("DispatcherMixer", 100), ("WindowAttention", 2500), ("SwiGLU", 100)])
def test_broadcast_inputs_in_inference(cls, T):
    layer = _layer(cls, torch.bfloat16)
    layer.use_fused_gates = layer.use_fused = True
    x = torch.randn(256, device=DEV).bfloat16().expand(2, T, 256)
    with torch.no_grad():
        assert torch.equal(layer(*_inputs(layer, cls, x)), layer(*_inputs(layer, cls, x.contiguous())))


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("cls", ["DispatcherMixer", "WindowAttention", "SwiGLU"])
def test_a_function_mode_sees_every_product(cls, train):
    from torch.overrides import TorchFunctionMode
    import torch.nn.functional as F
    layer = _layer(cls, torch.bfloat16)
    layer.use_fused_gates = layer.use_fused = True
    x = torch.randn(1, 100, 256, device=DEV).bfloat16()
    seen = []

    class Watch(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func is F.linear)
            return func(*args, **(kwargs or {}))

    with torch.set_grad_enabled(train):
        want = layer(*_inputs(layer, cls, x))
        with Watch():
            got = layer(*_inputs(layer, cls, x))
    assert sum(seen) == (3 if cls == "SwiGLU" else 4)
    assert (got.double() - want.double()).norm() <= 1e-2 * want.double().norm()


def test_gate_scan_without_a_gradient_says_so():
    """fused_gate_scan has no backward: with a gradient wanted, its result asks for one and refuses it."""
    from dispatcher_hybrid.fused_gates import fused_gate_scan
    b, T, H, L = 1, 40, 2, 5
    A, B, V0 = (torch.randn(b, T, 64 * H, device=DEV).bfloat16() for _ in range(3))
    W = [(torch.randn(L, H, 64 * H, device=DEV) * 0.05).bfloat16() for _ in range(3)]
    bias = [torch.zeros(L, H, device=DEV).bfloat16() for _ in range(3)]
    run = lambda: fused_gate_scan(A, B, *W, *bias, L, None, V0, H)
    want = run()
    for t in (A, W[1], bias[2], V0):
        t.requires_grad_()
        got = run()
        assert torch.equal(got, want) and got.requires_grad
        with pytest.raises(RuntimeError):
            got.sum().backward()
        with torch.no_grad():
            assert torch.equal(run(), want)
        t.requires_grad_(False)


def _last_dim_first(t):
    return t.movedim(-1, 0).contiguous().movedim(0, -1) if t.dim() > 1 else t


def _odd_offset(t):
    return torch.cat((t.flatten()[:1], t.flatten()))[1:].view(t.shape)


@pytest.mark.parametrize("unpack", [_last_dim_first, _odd_offset])
@pytest.mark.parametrize("cls,route", [("DispatcherMixer", "layer"), ("DispatcherMixer", "operation"),
                                       ("WindowAttention", "layer")])
def test_saved_tensors_may_come_back_in_another_layout(cls, route, unpack):
    """A saved-tensor hook that hands back the same values in other strides or at another alignment changes no gradient."""
    layer = _layer(cls, torch.bfloat16)
    layer.use_fused_gates = layer.use_fused = True
    if route == "operation":                                     # a hook on a projection: the gate path's registered operation
        layer.linear_in.register_forward_hook(lambda m, i, o: o * 1)
    x, dy = (torch.randn(2, 70, 256, device=DEV).bfloat16() for _ in range(2))
    x.requires_grad_()
    leaves = [x, *layer.parameters()]
    want = torch.autograd.grad(layer(*_inputs(layer, cls, x)), leaves, dy)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach().clone(), unpack):
        y = layer(*_inputs(layer, cls, x))
    for a, e in zip(torch.autograd.grad(y, leaves, dy), want):
        if route == "layer":
            assert torch.equal(a, e)
        else:                                                    # (library products of other layouts sum in other orders)
            assert (a.double() - e.double()).norm() <= 1e-2 * e.double().norm()


def test_training_runs_a_modules_own_scan_and_rotation():
    """A mixer with another gate activation and an attention layer with another rotation train with them (the torch path's
    output, tolerance as above)."""
    import dispatcher_hybrid.modeling_dispatcher as md
    mx, at = _layer("DispatcherMixer", torch.bfloat16), _layer("WindowAttention", torch.bfloat16)
    mx.activate = lambda i, f, r, m: md.DispatcherMixer.activate(i, f, r, 0.5 * m)
    at.apply_rope = lambda x, T: x
    x = torch.randn(1, 100, 256, device=DEV).bfloat16()
    for layer, cls in ((mx, "DispatcherMixer"), (at, "WindowAttention")):
        want = layer(*_inputs(layer, cls, x))
        layer.use_fused_gates = layer.use_fused = True
        got = layer(*_inputs(layer, cls, x))
        assert (got.double() - want.double()).norm() <= 1e-2 * want.double().norm()
        got.sum().backward()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("b,T,masked", [(1, 1, False), (1, 203, False), (2, 70, True), (3, 257, True), (3, 64, "shared"),
                                        (2, 1500, True)])
def test_one_call_mixer_layer_equals_its_launches(b, T, masked, dtype):
    """mixer_layer against fused_projections, fused_gate_scan and the output projection on their own, bit for bit."""
    from dispatcher_hybrid import fused_gates as fg
    mx = _layer("DispatcherMixer", dtype)
    L = mx.levels
    n_lv = min(L, T.bit_length())
    x = torch.randn(b, T, 256, device=DEV).to(dtype)
    mask = None
    if masked:
        mask = (torch.rand(1 if masked == "shared" else b, T, L, device=DEV) < 0.8).to(dtype)
    with torch.no_grad():
        weights = fg.mixer_layer_fits(mx, x)
        got = fg.mixer_layer(mx, x, mask, n_lv, weights)
        V0, A, B = fg.fused_projections(x, [mx.linear_in.weight, mx.gate_hidden.weight, mx.gate_hidden_src.weight])
        (Wi, bi), (Wf, bf), (Wr, br) = weights[0]
        m = None if mask is None else mask.expand(b, T, L)
        V = fg.fused_gate_scan(A, B, Wi, Wf, Wr, bi, bf, br, n_lv, m, V0, mx.num_heads)
        assert torch.equal(got, fg.fused_projections(V, [mx.linear_out.weight])[0])


@pytest.mark.parametrize("T", [100, 2500])
def test_attention_takes_a_hooked_projection_in_another_layout(T):
    layer = _layer("WindowAttention", torch.bfloat16)
    layer.linear_k.register_forward_hook(lambda m, i, o: 2 * torch.cat((o[..., :8], o), -1)[..., 8:])
    layer.linear_v.register_forward_hook(lambda m, i, o: _last_dim_first(o))
    x = torch.randn(2, T, 256, device=DEV).bfloat16()
    with torch.no_grad():
        want = layer(x)
        layer.use_fused = True
        got = layer(x)
    assert (got.double() - want.double()).norm() <= 1e-2 * want.double().norm()


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("moved", [_last_dim_first, _odd_offset])
def test_mixer_takes_hooked_projections_and_gate_weights_in_another_layout(moved, dtype, train):
    mx = _layer("DispatcherMixer", dtype)
    for l in (mx.linear_in, mx.gate_hidden, mx.gate_hidden_src):
        l.register_forward_hook(lambda m, i, o: moved(o))
    mx.forget_out.data = _odd_offset(mx.forget_out.data)
    x = torch.randn(2, 100, 256, device=DEV).to(dtype)
    with torch.set_grad_enabled(train):
        want = mx(*_inputs(mx, "DispatcherMixer", x))
        mx.use_fused_gates = True
        got = mx(*_inputs(mx, "DispatcherMixer", x))
    assert (got.double() - want.double()).norm() <= (1e-2 if dtype == torch.bfloat16 else 2e-5) * want.double().norm()
    if train:
        got.sum().backward()
        assert all(p.grad.isfinite().all() for p in mx.parameters())
