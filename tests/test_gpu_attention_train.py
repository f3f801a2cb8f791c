"""The attention layer's training pass (dh_window_attention_train_fwd / _bwd) against float64 autograd at the edges of its
64-row blocks and of the window. Tolerance (2-norm relative): projections, rotated rows (four roundings each), P and dS as
matrix operands, dO and the results are each rounded to bf16 (2^-9): at most ~10 roundings on any path, in quadrature
3.2 x 2^-9 = 6e-3; 1.5e-2 holds twice that."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _layer(d, window, max_len=4096):
    from dispatcher_hybrid import DispatcherConfig
    from dispatcher_hybrid.modeling_dispatcher import WindowAttention
    torch.manual_seed(d + window)
    at = WindowAttention(DispatcherConfig(d_model=d, num_heads=d // 64, max_len=max_len, attn_window=window, num_layers=1,
                                          vocab_size=64, dim_feedforward=64)).to(DEV, torch.bfloat16)
    with torch.no_grad():
        for p in at.parameters():
            p.normal_(std=1.5 / math.sqrt(d))
    at.use_fused = True
    return at


def _truth(at, x, dy):
    W = [l.weight.detach().double().requires_grad_() for l in (at.linear_q, at.linear_k, at.linear_v, at.linear_out)]
    x = x.detach().double().requires_grad_()
    b, T, d = x.shape
    H = at.num_heads
    cos, sin = (t.double() for t in at.rope_tables(T, x.device, torch.bfloat16))

    def rope(z):
        e, o = z[..., 0::2], z[..., 1::2]
        return torch.stack((e * cos - o * sin, e * sin + o * cos), -1).flatten(-2)

    q, k, v = ((x @ w.T).view(b, T, H, 64).transpose(1, 2) for w in W[:3])
    q, k = rope(q), rope(k)
    t = torch.arange(T, device=x.device)
    seen = t.unsqueeze(0) <= t.unsqueeze(1)
    if at.window > 0:
        seen &= t.unsqueeze(1) - t.unsqueeze(0) < at.window
    s = (q @ k.transpose(-2, -1).contiguous() / 8).masked_fill(~seen, float("-inf"))
    y = (torch.softmax(s, -1) @ v).transpose(1, 2).reshape(b, T, d) @ W[3].T
    y.backward(dy.double())
    return [y.detach(), x.grad] + [w.grad for w in W]


@pytest.mark.parametrize("b,T,d,window", [
    (1, 1, 64, 8), (2, 2, 128, 1), (1, 63, 64, 16), (1, 64, 192, 64), (2, 65, 64, 1000), (1, 128, 64, 0), (1, 129, 64, 33),
    (2, 200, 128, 64), (1, 321, 64, 65), (1, 700, 64, 128), (1, 1100, 128, 1024)])
def test_attention_train_against_float64(b, T, d, window):
    at = _layer(d, window)
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(b, T, d, device=DEV, generator=g).bfloat16().requires_grad_()
    dy = torch.randn(b, T, d, device=DEV, generator=g).bfloat16()
    ref = _truth(at, x, dy)
    y = at(x)
    assert "AttentionTrain" in y.grad_fn.name()
    y.backward(dy)
    got = [y.detach(), x.grad] + [l.weight.grad for l in (at.linear_q, at.linear_k, at.linear_v, at.linear_out)]
    for n, a, e in zip(["y", "dx", "dWq", "dWk", "dWv", "dWo"], got, ref):
        # a query that sees one key has no score gradient: what is left there is the rounding of dO . V - delta
        floor = 2.0 ** -8 * ref[4].norm() if n in ("dWq", "dWk") else 0.0
        assert (a.double() - e).norm() <= 1.5e-2 * e.norm() + floor, (n, ((a.double() - e).norm() / e.norm()).item())


def test_attention_train_matches_inference_and_reruns():
    at = _layer(128, 64)
    x = torch.randn(2, 190, 128, device=DEV).bfloat16()
    with torch.no_grad():
        inf = at(x)
    xg = x.clone().requires_grad_()
    outs = []
    for _ in range(2):
        y = at(xg)
        grads = torch.autograd.grad(y.float().square().sum(), [xg] + list(at.parameters()))
        outs.append([y.detach(), *grads])
    assert torch.equal(outs[0][0], inf)
    assert all(torch.equal(a, b) for a, b in zip(*outs))


def test_attention_train_other_dtypes_hooks_and_frozen_layers_keep_the_eager_path():
    at = _layer(64, 16)
    x = torch.randn(1, 40, 64, device=DEV).bfloat16()
    calls = []
    handle = at.linear_k.register_forward_hook(lambda m, i, o: calls.append(1))
    at(x)
    handle.remove()
    assert calls
    at32 = _layer(64, 16).float()
    x32 = x.float().requires_grad_()
    at32(x32).sum().backward()
    assert x32.grad.dtype == torch.float32
    at.requires_grad_(False)
    at.linear_v.weight.requires_grad_(True)
    at(x).sum().backward()
    assert at.linear_q.weight.grad is None and at.linear_v.weight.grad.isfinite().all()
