"""Which projections the fused inference layers multiply by their weights directly, and which they call, on the CPU."""

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
