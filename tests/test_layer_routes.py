"""What the fused layers hand to the kernels, on the CPU: the projections they multiply by directly and those they call, and
the layouts of their operands."""

from types import SimpleNamespace

import pytest
import torch
import torch.nn as nn


class Doubled(nn.Linear):
    def forward(self, h):
        return 2 * super().forward(h)


def _hooked(l):
    l.register_forward_hook(lambda m, i, o: 2 * o)
    return l


def _replaced(l):
    l.forward = lambda h: 2 * nn.Linear.forward(l, h)
    return l


def _offset(l):
    flat = torch.zeros(l.weight.numel() + 1, dtype=l.weight.dtype)        # a view of a flat buffer, rows not 16-byte aligned
    l.weight.data = flat[1:].view_as(l.weight)
    return l


NOT_PLAIN = {"hook": _hooked, "replaced forward": _replaced, "unaligned weight": _offset,
             "adapter": lambda l: Doubled(l.in_features, l.out_features, bias=False).to(l.weight.dtype),
             "bias": lambda l: nn.Linear(l.in_features, l.out_features).to(l.weight.dtype)}


@pytest.mark.parametrize("kind", NOT_PLAIN)
def test_only_plain_projections_are_multiplied_directly(kind):
    from dispatcher_hybrid import fused_gates as fg
    make = lambda: nn.Linear(64, 64, bias=False).bfloat16()
    x = SimpleNamespace(is_cuda=True, dtype=torch.bfloat16, shape=(1, 8, 64))         # what the predicates read of a GPU input
    assert fg.projections_fit(x, [make(), make()]) and fg.swiglu_fits(x, make(), make())
    assert not fg.projections_fit(x, [make(), NOT_PLAIN[kind](make())])
    assert not fg.swiglu_fits(x, NOT_PLAIN[kind](make()), make())
    assert not fg.swiglu_fits(x, make(), NOT_PLAIN[kind](make()))


def test_rows_a_kernel_cannot_read_are_copied():
    """Row operands of the products and their gradients: unit stride, rows at least a row apart, 16-byte aligned."""
    from dispatcher_hybrid.fused_gates import _rows16
    base = torch.arange(40 * 72, dtype=torch.float32).bfloat16().view(40, 72)
    kept = [base, base[:, :64], base[:, 8:72], base[::2], base.view(5, 8, 72)]
    copied = [base[0].expand(40, 72), base[:5, None].expand(5, 8, 72)[:, :, :64].reshape(5, 8, 64).transpose(0, 1),
              base[None, 0].expand(8, 40, 72), base[:, 1:65], base.view(-1)[1:65].view(1, 64), base.t(),
              base.view(-1)[:8 * 40 + 64].as_strided((41, 64), (8, 1)), base[:1, :66].as_strided((1, 64), (66, 1))]
    for t in kept:
        assert _rows16(t, 8).data_ptr() == t.data_ptr()
    for t in copied:
        r = _rows16(t, 8)
        assert torch.equal(r, t) and r.is_contiguous() and r.stride(-2) == t.shape[-1] and r.data_ptr() % 16 == 0
