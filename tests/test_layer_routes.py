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
    # what the predicates read of a GPU input
    x = SimpleNamespace(is_cuda=True, dtype=torch.bfloat16, shape=(1, 8, 64), device=torch.device("cpu"))
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


def _mixer(dtype=torch.bfloat16, d=64):
    from dispatcher_hybrid import DispatcherConfig
    from dispatcher_hybrid.modeling_dispatcher import DispatcherMixer
    torch.manual_seed(d)
    return DispatcherMixer(DispatcherConfig(d_model=d, num_heads=d // 64, max_len=64, num_layers=1, attn_layers=(),
                                            vocab_size=64, dim_feedforward=64)).to(dtype)


class _NoLibrary:
    def __getattr__(self, name):
        raise AssertionError(f"{name}: the library was reached")


def test_host_pointers_never_reach_a_kernel(monkeypatch):
    """Tensors that are not on the GPU, or not all on one, raise before any library call."""
    from dispatcher_hybrid import _hip
    from dispatcher_hybrid import fused_gates as fg
    from dispatcher_hybrid import fused_train as ft
    monkeypatch.setattr(_hip, "lib", _NoLibrary())
    mx, T, L = _mixer(), 8, 4
    (Wi, bi), (Wf, bf), (Wr, br) = [(w.detach(), b.detach()) for w, b in mx._gate_params()]
    A = torch.zeros(1, T, 64).bfloat16()
    mask, pre = torch.ones(1, T, L).bfloat16(), torch.zeros(1, T, L, 1).bfloat16()
    with torch.no_grad():
        for call in (lambda: fg.fused_gate_scan(A, A, Wi, Wf, Wr, bi, bf, br, L, mask, A, 1),
                     lambda: fg._scan_launch(pre, pre, pre, None, A, A, 1, L, 0, "scan"),
                     lambda: fg.mixer_layer(mx, A, mask, L, fg.plain_mixer_weights(mx, A.dtype, A.device)),
                     lambda: fg._preacts_bwd_launch(A, A, Wi, Wf, Wr, [pre] * 3, mask, [A, A], L, L, "bwd"),
                     lambda: ft._gate_scan_fwd(A, A, (Wi, Wf, Wr), (bi, bf, br), mask, A, 1, L, "train")):
            with pytest.raises(RuntimeError, match="GPU|device|Could not run"):
                call()
    on_gpu = SimpleNamespace(is_cuda=True, get_device=lambda: 0, device="cuda:0")
    _hip.same_gpu("x", on_gpu, None, on_gpu)
    with pytest.raises(RuntimeError, match="one device"):
        _hip.same_gpu("x", on_gpu, None, A)


def test_layers_and_masks_on_another_device_are_not_launched_directly():
    from dispatcher_hybrid import fused_gates as fg
    from dispatcher_hybrid import fused_train as ft
    mx, elsewhere = _mixer(), torch.device("meta")
    x = torch.zeros(1, 8, 64).bfloat16()
    mask = torch.ones(8, 6).bfloat16()
    assert fg.plain_linear(mx.linear_in, x.dtype, 64, x.device) and not fg.plain_linear(mx.linear_in, x.dtype, 64, elsewhere)
    with torch.no_grad():
        assert fg.mixer_layer_fits(mx, x) and not fg.mixer_layer_fits(mx, x.to(elsewhere))
    assert ft.mixer_fits(mx, x, mask, 4)
    assert not ft.mixer_fits(mx, x.to(elsewhere), mask.to(elsewhere), 4) and not ft.mixer_fits(mx, x, mask.to(elsewhere), 4)


def test_masks_of_other_sizes_raise_or_broadcast():
    from dispatcher_hybrid.fused_gates import _mask_view
    b, T, n = 2, 8, 3
    for shape in ((2, 8, 5), (2, 8, 3), (1, 8, 3), (1, 8, 5), (2, 1, 1)):
        mask = torch.rand(shape)
        m, *strides = _mask_view(mask, torch.float32, b, T, n)
        assert torch.equal(m.as_strided((b, T, n), strides), mask[..., :n].expand(b, T, n))
    for shape in ((2, 7, 3), (2, 8, 2), (3, 8, 3), (8, 3)):
        with pytest.raises((RuntimeError, ValueError)):
            _mask_view(torch.rand(shape), torch.float32, b, T, n)


def test_function_modes_see_a_layers_products():
    """Under a torch-function mode nothing is launched past it; a default device (a mode of torch's own) is not one."""
    from dispatcher_hybrid import fused_gates as fg
    from dispatcher_hybrid import fused_train as ft
    from torch.overrides import TorchFunctionMode

    class Watch(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    mx, x, mask = _mixer(), torch.zeros(1, 8, 64).bfloat16(), torch.ones(8, 6).bfloat16()
    gpu = SimpleNamespace(is_cuda=True, dtype=x.dtype, shape=x.shape, device=x.device)
    lin = mx.linear_in

    def routes():
        return [fg.plain_eager(), fg.projections_fit(gpu, [lin]), fg.swiglu_fits(gpu, lin, lin),
                fg.mixer_layer_fits(mx, x) is not None, ft.mixer_fits(mx, x, mask, 4) is not None]

    assert all(routes())
    with torch.device("cpu"):
        assert all(routes())
        with Watch():
            assert not any(routes())
    with Watch():
        assert not any(routes())


def test_saved_tensors_in_another_layout_are_copied_back():
    from dispatcher_hybrid.fused_train import _dense
    t = torch.arange(120.).view(2, 3, 20)
    assert _dense(t).data_ptr() == t.data_ptr()
    for other in (t.transpose(0, 2).contiguous().transpose(0, 2), torch.cat((t[..., :1], t), -1)[..., 1:],
                  torch.cat((torch.zeros(1), t.flatten()))[1:].view_as(t)):
        d = _dense(other)
        assert torch.equal(d, t) and d.is_contiguous() and d.data_ptr() % 16 == 0


def test_methods_of_a_subclass_or_an_instance_are_seen():
    from dispatcher_hybrid.modeling_dispatcher import DispatcherMixer, _replaced

    class Named(DispatcherMixer):
        pass

    class Gentle(Named):
        @staticmethod
        def activate(pre_i, pre_f, pre_r, m):
            return DispatcherMixer.activate(pre_i, pre_f, pre_r, 0.5 * m)

    mx, names = _mixer(), ("_scan_eager", "activate")
    assert not _replaced(mx, DispatcherMixer, names)
    for cls, other in ((Named, False), (Gentle, True)):
        mx.__class__ = cls
        assert _replaced(mx, DispatcherMixer, names) is other
    mx.__class__ = DispatcherMixer
    mx.activate = Gentle.activate
    assert _replaced(mx, DispatcherMixer, names)
