"""dispatcher::gate_scan_train (pre-activations + level scan with one backward) against float64 autograd of the eager
mixer's formula, at the edges of its tiles: 64-position tiles with a 63-position halo, levels 0-5 inside a tile, levels
6-11 along residue classes mod 64 of at most 16 / 32 / 64 positions.

Tolerances (2-norm relative). fp32: sums of at most a few thousand terms and 12 levels of fp32 updates, and the hardware
exponential's 1 ulp: 2e-5 bounds 12 levels x ~2^-20. bf16: pre-activations, states and their gradients are each rounded once
per level (2^-9 relative), 12 levels and 3 roundings each in quadrature ~ 6 x 2^-9 = 1.2e-2; 2.5e-2 holds twice that."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _truth(A, B, W, bias, mask, V0, dV, H, n_lv):
    leaves = [t.detach().double().requires_grad_() for t in (A, B, *W, *bias, V0)]
    A, B, Wi, Wf, Wr, bi, bf, br, V0 = leaves
    b, T, d = V0.shape
    V = V0.view(b, T, H, d // H)
    m_all = mask.double().expand(b, T, mask.shape[-1])
    t = torch.arange(T, device=DEV)
    for l in range(n_lv):
        lag = 1 << l
        src = lambda x: torch.cat([torch.zeros_like(x[:, :min(lag, T)]), x[:, :max(T - lag, 0)]], 1)
        m = m_all[..., l:l + 1] * (t >= lag).view(1, T, 1)
        hid = torch.relu(A + src(B) * (m > 0 if mask.dim() == 3 else (t >= lag).view(1, T, 1))) ** 2
        si, sf, sr = (torch.sigmoid(hid @ w[l].T + c[l]) for w, c in ((Wi, bi), (Wf, bf), (Wr, br)))
        V = (sf * m + 1 - m).unsqueeze(-1) * V + (si * m).unsqueeze(-1) * src(sr.unsqueeze(-1) * V)
    V = V.reshape(b, T, d)
    V.backward(dV.double())
    return [V.detach()] + [x.grad for x in leaves]


CASES = [  # b, T, H, mask kind ("level", "doc", "soft": fractional values)
    (1, 1, 1, "level"), (2, 2, 3, "doc"), (1, 63, 4, "doc"), (1, 64, 5, "soft"), (2, 65, 2, "doc"), (1, 127, 1, "level"),
    (3, 129, 4, "soft"), (1, 777, 3, "level"), (2, 1024, 2, "doc"), (1, 1025, 2, "doc"), (1, 2048, 1, "level"),
    (1, 2049, 5, "doc"), (1, 4095, 1, "doc"), (1, 4096, 2, "doc")]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,T,H,kind", CASES)
def test_gate_scan_train_against_float64(b, T, H, kind, dtype):
    from dispatcher_hybrid.fused_train import gate_scan_train
    g = torch.Generator(device=DEV).manual_seed(T + H)
    rn = lambda *s: torch.randn(*s, device=DEV, generator=g)
    d, L = 64 * H, 12
    n_lv = min(L, T.bit_length())
    A, B, V0 = (rn(b, T, d).mul(0.6).to(dtype) for _ in range(3))
    W = [(rn(L, H, d) * 0.05).to(dtype) for _ in range(3)]
    bias = [torch.full((L, H), c, device=DEV).add(rn(L, H) * 0.1).to(dtype) for c in (-1.0, 1.5, 2.0)]
    lag = 1 << torch.arange(L, device=DEV)
    t = torch.arange(T, device=DEV).unsqueeze(1)
    mask = ((t >= lag) & (lag < T)).to(dtype)
    if kind != "level":
        mask = mask * (torch.rand(b, T, L, device=DEV, generator=g) < 0.9)
    if kind == "soft":
        mask = mask * (0.5 + 0.5 * torch.rand(b, T, L, device=DEV, generator=g)).to(dtype)
    dV = rn(b, T, d).to(dtype)
    ref = _truth(A, B, W, bias, mask, V0, dV, H, n_lv)
    leaves = [x.clone().requires_grad_() for x in (A, B, *W, *bias, V0)]
    V = gate_scan_train(leaves[0], leaves[1], *leaves[2:8], n_lv, mask, leaves[8], H)
    V.backward(dV)
    got = [V.detach()] + [x.grad for x in leaves]
    names = ["V", "dA", "dB", "dWi", "dWf", "dWr", "dbi", "dbf", "dbr", "dV0"]
    for n, x, y in zip(names, got, ref):
        assert x.dtype == dtype and x.shape == y.shape
        err, size = (x.double() - y).norm().item(), y.norm().item()
        assert err <= (2e-5 if dtype == torch.float32 else 2.5e-2) * size + 1e-30, (n, err / max(size, 1e-30))


def test_gate_scan_train_matches_module_fallback():
    """The mixer's training pass through the operation and through the torch scan (a mask that takes gradients keeps it
    there) give the same fp32 output and gradients."""
    from dispatcher_hybrid import DispatcherConfig
    from dispatcher_hybrid.modeling_dispatcher import DispatcherMixer
    torch.manual_seed(3)
    cfg = DispatcherConfig(d_model=128, num_heads=2, max_len=256, num_layers=1, attn_layers=(), vocab_size=64,
                           dim_feedforward=128)
    mx = DispatcherMixer(cfg).to(DEV)
    with torch.no_grad():
        for p in mx.parameters():
            if p.dim() > 1 and p.shape != (8, 2):
                p.normal_(std=0.1)
    mx.use_fused_gates = True
    x0 = torch.randn(2, 150, 128, device=DEV)
    t = torch.arange(150, device=DEV).unsqueeze(1)
    mask = (t >= (1 << torch.arange(8, device=DEV))).float()
    outs = []
    for m in (mask, mask.clone().requires_grad_()):
        x = x0.clone().requires_grad_()
        mx.zero_grad()
        y = mx(x, m)
        y.square().sum().backward()
        outs.append([y.detach(), x.grad] + [p.grad.clone() for p in mx.parameters()])
    for a, b in zip(*outs):
        assert (a - b).norm() <= 2e-5 * b.norm()


def test_gate_scan_train_under_checkpoint_and_autocast():
    """Activation checkpointing recomputes the operation; under autocast (bf16 activations, fp32 weights) the weights'
    gradients come back in fp32."""
    from dispatcher_hybrid.fused_train import gate_scan_train
    from torch.utils.checkpoint import checkpoint
    g = torch.Generator(device=DEV).manual_seed(1)
    b, T, H, L = 1, 100, 2, 7
    A, B, V0 = (torch.randn(b, T, 64 * H, device=DEV, generator=g).bfloat16().requires_grad_() for _ in range(3))
    W = [(torch.randn(L, H, 64 * H, device=DEV, generator=g) * 0.05).requires_grad_() for _ in range(3)]
    bias = [torch.zeros(L, H, device=DEV).requires_grad_() for _ in range(3)]
    mask = (torch.arange(T, device=DEV).unsqueeze(1) >= (1 << torch.arange(L, device=DEV))).float()
    leaves = [A, B, *W, *bias, V0]
    f = lambda *xs: gate_scan_train(*xs[:8], L, mask, xs[8], H)
    plain = torch.autograd.grad(f(*leaves).float().square().sum(), leaves)
    again = torch.autograd.grad(checkpoint(f, *leaves, use_reentrant=False).float().square().sum(), leaves)
    assert all(p.dtype == x.dtype for p, x in zip(plain, leaves))
    assert all(torch.equal(p, q) for p, q in zip(plain, again))


def _mixer(dtype, d=128, max_len=256):
    from dispatcher_hybrid import DispatcherConfig
    from dispatcher_hybrid.modeling_dispatcher import DispatcherMixer
    torch.manual_seed(5)
    mx = DispatcherMixer(DispatcherConfig(d_model=d, num_heads=d // 64, max_len=max_len, num_layers=1, attn_layers=(),
                                          vocab_size=64, dim_feedforward=128)).to(DEV, dtype)
    with torch.no_grad():
        for n, p in mx.named_parameters():
            if "bias" not in n:
                p.normal_(std=0.08)
    return mx


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-5), (torch.bfloat16, 2.5e-2)])
@pytest.mark.parametrize("b,T", [(1, 1), (2, 65), (3, 256)])
def test_mixer_train_against_float64_eager(b, T, dtype, tol):
    """The whole-layer operation against the eager mixer in float64 (tolerances as above)."""
    mx = _mixer(dtype)
    ref = _mixer(torch.float64)
    ref.load_state_dict({n: p.double() for n, p in mx.state_dict().items()})
    mx.use_fused_gates = True
    t = torch.arange(T, device=DEV).unsqueeze(1)
    lag = 1 << torch.arange(8, device=DEV)
    mask = ((t >= lag) & (lag < T)).to(dtype)
    x = torch.randn(b, T, 128, device=DEV).to(dtype).requires_grad_()
    x64 = x.detach().double().requires_grad_()
    dy = torch.randn(b, T, 128, device=DEV).to(dtype)
    y, y64 = mx(x, mask), ref(x64, mask.double())
    y.backward(dy)
    y64.backward(dy.double())
    pairs = [("y", y, y64), ("dx", x.grad, x64.grad)]
    pairs += [(n, p.grad, q.grad) for (n, p), q in zip(mx.named_parameters(), ref.parameters())]
    for n, a, e in pairs:
        assert a.dtype == dtype
        assert (a.double() - e).norm() <= tol * e.norm() + 1e-30, (n, ((a.double() - e).norm() / e.norm()).item())


def test_mixer_train_partial_gradients_hooks_and_adapters():
    """Frozen inputs or weights get no gradient; a hooked or replaced projection keeps being called."""
    mx = _mixer(torch.float32)
    mx.use_fused_gates = True
    t = torch.arange(40, device=DEV).unsqueeze(1)
    mask = (t >= (1 << torch.arange(8, device=DEV))).float()
    x = torch.randn(1, 40, 128, device=DEV)
    full = mx(x, mask)
    full.sum().backward()
    want = {n: p.grad.clone() for n, p in mx.named_parameters()}
    mx.zero_grad()
    for n, p in mx.named_parameters():
        p.requires_grad_(n in ("gate_out", "reset_out_bias"))
    mx(x, mask).sum().backward()
    assert mx.linear_in.weight.grad is None
    assert torch.equal(mx.gate_out.grad, want["gate_out"]) and torch.equal(mx.reset_out_bias.grad, want["reset_out_bias"])
    mx.requires_grad_(True)
    calls = []
    handle = mx.gate_hidden.register_forward_hook(lambda m, i, o: calls.append(1))
    hooked = mx(x, mask)
    handle.remove()
    assert calls and (hooked - full).norm() <= 2e-5 * full.norm()

    class Adapter(torch.nn.Linear):
        def forward(self, h):
            return 2 * super().forward(h)

    ad = Adapter(128, 128, bias=False).to(DEV)
    ad.weight = mx.linear_out.weight
    mx.linear_out = ad
    assert (mx(x, mask) - 2 * full).norm() <= 4e-5 * full.norm()


def test_mixer_train_under_transforms():
    """A saved-tensor hook sees what the whole-layer operation keeps; torch.func transforms (which registered operations do
    not take) and second derivatives are refused, not silently wrong; a compiler gets the layer-by-layer form and the same
    gradients."""
    mx = _mixer(torch.float32)
    mx.use_fused_gates = True
    t = torch.arange(70, device=DEV).unsqueeze(1)
    mask = (t >= (1 << torch.arange(8, device=DEV))).float()
    x = torch.randn(1, 70, 128, device=DEV)
    xg = x.clone().requires_grad_()
    want, = torch.autograd.grad(mx(xg, mask).square().sum(), xg)
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda z: mx(z, mask).square().sum())(x)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda z: packed.append(z.numel()) or z.cpu(), lambda z: z.to(DEV)):
        loss = mx(xg, mask).square().sum()
    hooked, = torch.autograd.grad(loss, xg)
    assert packed and torch.equal(hooked, want)
    g1, = torch.autograd.grad(mx(xg, mask).square().sum(), xg, create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(g1.sum(), xg)
    compiled = torch.compile(mx, backend="aot_eager", fullgraph=True)
    traced, = torch.autograd.grad(compiled(xg, mask).square().sum(), xg)
    assert (traced - want).norm() <= 2e-5 * want.norm()


@pytest.mark.parametrize("T", [24, 100, 200, 256, 257, 500])
def test_mixer_train_fp32_is_as_exact_as_layer_by_layer(T):
    """Distance from float64 of the whole-layer operation's fp32 output and gradients against that of the layer-by-layer
    form (torch products and scan; a mask that takes gradients keeps it there), whose sums are no longer than 1024 terms:
    at most 1.15 times it, which covers the other order of the same sums."""
    mx, ref = _mixer(torch.float32, 1024, 512), _mixer(torch.float64, 1024, 512)
    with torch.no_grad():
        for n, p in mx.named_parameters():
            if "bias" not in n:
                p.mul_(0.25)
    ref.load_state_dict({n: p.double() for n, p in mx.state_dict().items()})
    mx.use_fused_gates = True
    t = torch.arange(T, device=DEV).unsqueeze(1)
    mask = (t >= (1 << torch.arange(9, device=DEV))).float()
    g = torch.Generator(device=DEV).manual_seed(2)
    x, dy = (torch.randn(1, T, 1024, device=DEV, generator=g) for _ in range(2))

    def grads(layer, x, m, dy):
        x = x.clone().requires_grad_()
        layer.zero_grad()
        y = layer(x, m)
        y.backward(dy)
        return [("y", y.detach()), ("dx", x.grad)] + [(n, p.grad.clone()) for n, p in layer.named_parameters()]

    exact = grads(ref, x.double(), mask.double(), dy.double())
    whole, parts = grads(mx, x, mask, dy), grads(mx, x, mask.clone().requires_grad_(), dy)
    for (n, e), (_, a), (_, b) in zip(exact, whole, parts):
        if "bias" not in n:                                      # (a few hundred values: their distance is a matter of luck)
            assert (a.double() - e).norm() <= 1.15 * (b.double() - e).norm(), n


def test_gate_scan_train_fp32_far_gates():
    """Gates far from the middle: admit pre-activations of -85 .. -20 (a bias alone, exact) and their gradients, value by
    value. The library exp and an IEEE divide are within 2 ulp, the gradient's few products half of one each: 8 x 2^-24."""
    from dispatcher_hybrid.fused_train import gate_scan_train
    b, T, H, L = 1, 600, 1, 10
    A, B, V0 = torch.zeros(b, T, 64, device=DEV), torch.zeros(b, T, 64, device=DEV), torch.ones(b, T, 64, device=DEV)
    W = [torch.zeros(L, H, 64, device=DEV) for _ in range(3)]
    far = -torch.linspace(20, 85, L, device=DEV).view(L, H)
    bias = [far.clone().requires_grad_(), torch.full((L, H), 60.0, device=DEV), torch.full((L, H), 60.0, device=DEV)]
    mask = (torch.arange(T, device=DEV).unsqueeze(1) >= (1 << torch.arange(L, device=DEV))).float()
    V = gate_scan_train(A, B, *W, *bias, L, mask, V0, H)
    only = torch.zeros_like(V)
    only[0, T - 1, 0] = 1                                        # one destination: no sum over positions
    got, = torch.autograd.grad(V, bias[0], only)
    want = torch.sigmoid(far.double())                           # forget = transmit = V = 1 to 1e-9: d/dx sigmoid = itself
    assert ((got.double() - want).abs() <= 8 * 2.0 ** -24 * want).all()


@pytest.mark.parametrize("wide", [(6,), (3,), (4, 7)])
def test_gate_scan_train_keeps_wider_parameters_gradients(wide):
    """bf16 activations with some fp32 gate weights or biases: those parameters' gradients are the fp32 sums, not their bf16
    rounding, and the others round the same sums."""
    from dispatcher_hybrid.fused_train import gate_scan_train
    g = torch.Generator(device=DEV).manual_seed(4)
    b, T, H, L = 2, 150, 2, 8
    A, B, V0 = (torch.randn(b, T, 64 * H, device=DEV, generator=g).bfloat16() for _ in range(3))
    P = [(torch.randn(L, H, 64 * H, device=DEV, generator=g) * 0.05).bfloat16() for _ in range(3)]
    P += [torch.randn(L, H, device=DEV, generator=g).bfloat16() for _ in range(3)]
    mask = (torch.arange(T, device=DEV).unsqueeze(1) >= (1 << torch.arange(L, device=DEV))).float()
    dV = torch.randn(b, T, 64 * H, device=DEV, generator=g).bfloat16()

    def grads(fp32):
        leaves = [(p.float() if i + 2 in fp32 else p).clone().requires_grad_() for i, p in enumerate(P)]
        return torch.autograd.grad(gate_scan_train(A, B, *leaves, L, mask, V0, H), leaves, dV)

    full = grads(range(2, 8))
    for i, (p, f) in enumerate(zip(grads(wide), full)):
        if i + 2 in wide:
            assert p.dtype == torch.float32 and torch.equal(p, f) and not torch.equal(p, p.bfloat16().float())
        else:
            assert torch.equal(p, f.bfloat16())


@pytest.mark.parametrize("route", ["layer", "operation"])
def test_mixer_gradients_of_gradients_that_avoid_the_gate_readouts(route):
    """A penalty on the gradients of the value and output projections can be differentiated (through the scan, against the
    eager mixer in float64); one that needs second derivatives of the gate readouts is refused. fp32, 12 levels of updates in
    each direction: 5e-5."""
    mx, ref = _mixer(torch.float32), _mixer(torch.float64)
    ref.load_state_dict({n: p.double() for n, p in mx.state_dict().items()})
    mx.use_fused_gates = True
    if route == "operation":
        mx.linear_in.register_forward_hook(lambda m, i, o: o * 1)
    T = 70
    mask = (torch.arange(T, device=DEV).unsqueeze(1) >= (1 << torch.arange(8, device=DEV))).float()
    g = torch.Generator(device=DEV).manual_seed(6)
    x, dy = (torch.randn(2, T, 128, device=DEV, generator=g) for _ in range(2))

    def penalty(layer, x, m, dy):
        first = torch.autograd.grad(layer(x, m), [layer.linear_in.weight, layer.linear_out.weight], dy, create_graph=True)
        return [*first, *torch.autograd.grad(sum(f.square().sum() for f in first), list(layer.parameters()))]

    for a, e in zip(penalty(mx, x, mask, dy), penalty(ref, x.double(), mask.double(), dy.double())):
        assert (a.double() - e).norm() <= 5e-5 * e.norm()
    first, = torch.autograd.grad(mx(x, mask), mx.gate_hidden.weight, dy, create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(first.square().sum(), mx.gate_out)
