"""Which calls the directly launched training layers take, and the attention layer's twice-differentiable gradients, on the
CPU."""

import torch
import torch.autograd.forward_ad as fwad
import torch.nn as nn
from torch.utils.flop_counter import FlopCounterMode


def _attention(d=128, window=5):
    from dispatcher_hybrid import DispatcherConfig
    from dispatcher_hybrid.modeling_dispatcher import WindowAttention
    torch.manual_seed(d)
    return WindowAttention(DispatcherConfig(d_model=d, num_heads=d // 64, max_len=64, attn_window=window, num_layers=1,
                                            vocab_size=64, dim_feedforward=64))


def test_direct_launches_only_in_plain_eager_execution():
    from dispatcher_hybrid.fused_gates import plain_eager
    seen = []

    def probe(t):
        seen.append(plain_eager())
        return t * 1.0

    x = torch.ones(2, 3)
    probe(x)
    torch.func.vmap(probe)(x)
    with fwad.dual_level():
        probe(fwad.make_dual(x, x))
    with FlopCounterMode(display=False):
        probe(x)
    torch.jit.trace(probe, (x,), check_trace=False)
    probe(x)
    assert seen == [True, False, False, False, False, True]


def test_layers_with_something_around_their_product_are_not_plain():
    from dispatcher_hybrid.fused_gates import plain_linear
    plain = lambda l: plain_linear(l, torch.float32, 64)
    l = nn.Linear(64, 64, bias=False)
    assert plain(l)
    for register in (l.register_forward_hook, l.register_forward_pre_hook, l.register_full_backward_hook):
        handle = register(lambda *a: None)
        assert not plain(l)
        handle.remove()
    handle = nn.modules.module.register_module_forward_hook(lambda *a: None)
    assert not plain(l)
    handle.remove()
    assert plain(l)
    l.forward = l.forward                                        # replaced on the instance, as offloading wrappers do
    assert not plain(l)


def test_attention_gradients_can_be_differentiated_again():
    """Gradients and a gradient penalty's gradients against float64 autograd over the eager layer; two weights tied. fp32
    sums of at most 128 terms and a few chained products: 2e-5 relative."""
    from dispatcher_hybrid.fused_train import _attention_grads
    at = _attention()
    T, band = 23, at.band(23)
    cos, sin = at.rope_tables(T, torch.device("cpu"), torch.float32)
    g = torch.Generator().manual_seed(1)
    x, dy = (torch.randn(2, T, 128, generator=g) for _ in range(2))
    W = [torch.randn(128, 128, generator=g) / 11 for _ in range(3)]
    W = [W[0], W[0], W[1], W[2]]                                 # query and key weights are one tensor

    def both(dtype, grads):
        ins = [t.to(dtype).requires_grad_() for t in (x, W[0], W[2], W[3])]
        args = (ins[0], ins[1], ins[1], ins[2], ins[3])
        first = grads(args, dy.to(dtype))
        penalty = sum(v.square().sum() for v in first)
        return [*first, *torch.autograd.grad(penalty, ins)]

    def ours(args, d):
        gx, gq, gk, gv, go = _attention_grads(args, (True,) * 5, d, cos, sin, 2, band)
        return [gx, gq + gk, gv, go]

    def truth(args, d):
        a64 = _attention().double()
        a64._rope_cache[(T, torch.device("cpu"), torch.float64)] = (cos.double(), sin.double())
        y = torch.func.functional_call(a64, {"linear_%s.weight" % n: w for n, w in zip(("q", "k", "v", "out"), args[1:])},
                                       (args[0],))
        return list(torch.autograd.grad(y, [args[0], args[1], args[3], args[4]], d, create_graph=True))

    for a, e in zip(both(torch.float32, ours), both(torch.float64, truth)):
        assert (a.double() - e).norm() <= 2e-5 * e.norm()
