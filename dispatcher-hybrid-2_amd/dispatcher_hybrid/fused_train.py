"""Training passes of the fused layers on gfx950 kernels, each one operation with one backward.

    dispatcher::gate_scan_train   gate pre-activations + level scan (from the projections A, B, V0)
    mixer_train                   a whole mixer layer: projections, gate path, output projection
    attention_train               a whole sliding-window attention layer (bf16, 64-wide heads)

They run under ``model.enable_fused_gates()`` when gradients are wanted (DispatcherMixer picks the widest one that fits)
and replace the reference's eager autograd of the level loop and the attention (reference
dispatcher_hybrid/modeling_dispatcher.py:86-121, 163-182) and its fused gate op's backward (reference
dispatcher_hybrid/fused_gates.py:96-173, 225-257). Kernels: ``dh_gate_preacts_fwd``, ``dh_level_scan_train_fwd`` / ``_bwd``,
``dh_gate_preacts_bwd_ws``, ``dh_window_attention_train_fwd``, ``dh_window_attention_bwd``, ``dh_wgrad_gemm`` and, for the
plain products, ``dh_proj_gemm`` or the library.

Importing this module loads the kernel library and raises ImportError if it is missing.
"""

import ctypes
from types import SimpleNamespace
from typing import List

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import _hip
from .fused_gates import (OUT_GEMM_MAX_ROWS, PROJ_GEMM_MAX_ROWS, _preacts_bwd_launch, _preacts_launch, _rows16,
                          fused_gate_preacts, plain_eager, plain_mixer_weights, plain_square_weights,
                          projections_launch)

SCAN_MAX_LEN = 4096
SCAN_MAX_LEVELS = 12
SCAN_HEAD = 64


def scan_fits(A, B, V0, mask, num_heads, n_lv):
    """Whether the training scan takes these: fp32 or bf16 throughout, 64-wide heads (a wave holds a head's columns), at
    most 4096 positions and 12 levels, and a mask no gradient flows to."""
    return (A.dtype in (torch.float32, torch.bfloat16) and B.dtype == A.dtype and V0.dtype == A.dtype
            and V0.shape[-1] == SCAN_HEAD * num_heads and V0.shape[1] <= SCAN_MAX_LEN
            and n_lv <= SCAN_MAX_LEVELS and not mask.requires_grad)


def _gate_rows(b, H, n_lv, T, like):
    """Three head-major gate tensors (b, H, n_lv, T) in one allocation, rows padded to a multiple of 8 positions."""
    return torch.empty(3, b, H, n_lv, -(-T // 8) * 8, device=like.device, dtype=like.dtype)


def _scan_mask(mask, b, T, n_lv, cd):
    """The level (T, L) or document (b, T, L) mask as a (b, T, n_lv) view in dtype cd (other sizes raise)."""
    return mask[..., :n_lv].to(cd).expand(b, T, n_lv)


def _dense(t):
    """A saved tensor in the layout it was saved in, contiguous and 16-byte aligned (a saved-tensor hook may hand back
    another one)."""
    return t if t.is_contiguous() and t.data_ptr() % 16 == 0 else t.clone(memory_format=torch.contiguous_format)


def _gate_scan_fwd(A, B, W, bias, mask, V0, H, n_lv, what):
    """(V, pre, states) of the gate path; A, B, V0 (b, T, .) with unit-stride, 16-byte aligned rows, A and B alike."""
    b, T, d = V0.shape
    cd, dev = A.dtype, A.device
    _hip.same_gpu(what, V0, mask)                                              # (the others at the first launch)
    V = torch.empty(b, T, d, device=dev, dtype=cd)
    pre = _gate_rows(b, H, n_lv, T, A)
    states = torch.empty(n_lv - 1, b, T, d, device=dev, dtype=cd)
    bd = cd if all(v.dtype == cd for v in bias) else torch.float32             # (other biases: fp32 copies)
    W = [_rows16(w[:n_lv].contiguous().to(cd), 8) for w in W]
    bias = [v[:n_lv].contiguous().to(bd) for v in bias]
    m = _scan_mask(mask, b, T, n_lv, cd)
    gates = [g[..., :T].permute(0, 3, 2, 1) for g in pre]                      # logical (b, T, n_lv, H)
    _preacts_launch(A, B, *W, *bias, m if mask.dim() == 3 else None, gates, gates[0].stride(), 0,
                    n_lv, what)
    p = _hip.ptr
    st = _hip.lib.dh_level_scan_train_fwd(
        _hip.dtype_code(cd), p(pre[0]), p(pre[1]), p(pre[2]), pre.stride(1), pre.stride(3), pre.stride(2), p(m),
        *m.stride(), p(V0), V0.stride(0), V0.stride(1), p(states), p(V), b, T, H, d // H, n_lv, _hip.stream_handle(dev))
    _hip.check(st, what)
    return V, pre, states


def _gate_scan_bwd(A, B, W, mask, V0, pre, states, dV, dV0, outs, H, n_lv, what):
    """Fills dV0 and outs = [dA, dB, dWi, dWf, dWr, dbi, dbf, dbr] from dV; A, B, V0 as _gate_scan_fwd had them, dV0, dA, dB
    with unit-stride, 16-byte aligned rows."""
    b, T, d = V0.shape
    cd = A.dtype
    _hip.same_gpu(what, V0, mask, pre, states, dV)                             # (the others at the second launch)
    m, pre, states = _scan_mask(mask, b, T, n_lv, cd), _dense(pre), _dense(states)
    dpre = torch.empty_like(pre)
    scratch = torch.empty(b, T, d, device=A.device, dtype=cd)
    p = _hip.ptr
    st = _hip.lib.dh_level_scan_train_bwd(
        _hip.dtype_code(cd), p(pre[0]), p(pre[1]), p(pre[2]), pre.stride(1), pre.stride(3), pre.stride(2), p(m),
        *m.stride(), p(V0), V0.stride(0), V0.stride(1), p(states), p(dV), dV.stride(0), dV.stride(1), p(scratch), p(dV0),
        dV0.stride(0), dV0.stride(1), p(dpre[0]), p(dpre[1]), p(dpre[2]), b, T, H, d // H, n_lv,
        _hip.stream_handle(A.device))
    _hip.check(st, what)
    _preacts_bwd_launch(A, B, *W, [g[..., :T].permute(0, 3, 2, 1) for g in dpre], m if mask.dim() == 3 else None, outs,
                        n_lv, W[0].shape[0], what)


def _gate_grads(W, gh, od, dev):
    L, H = W.shape[:2]
    return ([torch.empty(L, H, gh, device=dev, dtype=od) for _ in range(3)]
            + [torch.empty(L, H, device=dev, dtype=od) for _ in range(3)])


# ---------------------------------------------------------------------------------------------
# dispatcher::gate_scan_train
# ---------------------------------------------------------------------------------------------
@torch.library.custom_op("dispatcher::gate_scan_train", mutates_args=(), device_types="cuda")
def _gate_scan_train_op(A: torch.Tensor, B: torch.Tensor, Wi: torch.Tensor, Wf: torch.Tensor, Wr: torch.Tensor,
                        bi: torch.Tensor, bf: torch.Tensor, br: torch.Tensor, mask: torch.Tensor, V0: torch.Tensor,
                        num_heads: int, n_lv: int) -> List[torch.Tensor]:
    b, T, d = V0.shape
    if b == 0 or T == 0:
        return [torch.empty_like(V0, memory_format=torch.contiguous_format), _gate_rows(b, num_heads, n_lv, T, A),
                A.new_empty(n_lv - 1, b, T, d)]
    A, B, V0 = (_rows16(t.contiguous(), 8) for t in (A, B, V0))
    return list(_gate_scan_fwd(A, B, (Wi, Wf, Wr), (bi, bf, br), mask, V0, num_heads, n_lv, "dispatcher::gate_scan_train"))


@_gate_scan_train_op.register_fake
def _(A, B, Wi, Wf, Wr, bi, bf, br, mask, V0, num_heads, n_lv):
    b, T, d = V0.shape
    return [torch.empty_like(V0, memory_format=torch.contiguous_format), _gate_rows(b, num_heads, n_lv, T, A),
            A.new_empty(n_lv - 1, b, T, d)]


@torch.library.custom_op("dispatcher::gate_scan_train_bwd", mutates_args=(), device_types="cuda")
def _gate_scan_train_bwd_op(A: torch.Tensor, B: torch.Tensor, Wi: torch.Tensor, Wf: torch.Tensor, Wr: torch.Tensor,
                            mask: torch.Tensor, V0: torch.Tensor, pre: torch.Tensor, states: torch.Tensor,
                            dV: torch.Tensor, num_heads: int, n_lv: int, wide: bool) -> List[torch.Tensor]:
    # the gradients in A's dtype, or (wide: wider weights or biases, as under autocast) in fp32
    od = torch.float32 if wide else A.dtype
    dV0 = torch.empty(V0.shape, device=A.device, dtype=A.dtype)
    outs = [torch.empty(A.shape, device=A.device, dtype=od) for _ in range(2)] + _gate_grads(Wi, A.shape[-1], od, A.device)
    if V0.numel() == 0:
        return [dV0] + [o.zero_() for o in outs]
    A, B, V0, dV = (_rows16(t.contiguous(), 8) for t in (A, B, V0, dV.to(A.dtype)))
    _gate_scan_bwd(A, B, (Wi, Wf, Wr), mask, V0, pre, states, dV, dV0, outs, num_heads, n_lv,
                   "dispatcher::gate_scan_train_bwd")
    return [dV0] + outs


@_gate_scan_train_bwd_op.register_fake
def _(A, B, Wi, Wf, Wr, mask, V0, pre, states, dV, num_heads, n_lv, wide):
    od = torch.float32 if wide else A.dtype
    return ([A.new_empty(V0.shape)] + [A.new_empty(A.shape, dtype=od) for _ in range(2)]
            + _gate_grads(Wi, A.shape[-1], od, A.device))


def _scan_again(A, B, Wi, Wf, Wr, bi, bf, br, V0, mask, H, n_lv):
    """The gate path as torch operations after fused_gate_preacts: differentiable twice in all but the pre-activations (whose
    operation refuses that), as the layer was before it had a backward of its own."""
    from .modeling_dispatcher import DispatcherMixer
    b, T, d = V0.shape
    m3 = mask[..., :n_lv].expand(b, T, n_lv) if mask.dim() == 3 else None
    pre = fused_gate_preacts(A, B, Wi, Wf, Wr, bi, bf, br, n_lv, m3)
    mx = SimpleNamespace(num_heads=H, shifts=[1 << l for l in range(n_lv)], activate=DispatcherMixer.activate,
                         level_update=DispatcherMixer.level_update)
    _, m_heads = DispatcherMixer._masks(mx, mask, b, T, n_lv)
    V = V0.view(b, T, H, d // H).transpose(1, 2).reshape(b * H, T, d // H)
    V = DispatcherMixer._scan_eager(mx, V, *pre, m_heads.to(V.dtype), b, T, n_lv)
    return V.view(b, H, T, d // H).transpose(1, 2).reshape(b, T, d)


def _grads_again(out, inputs, need, dout):
    """The gradients of `inputs` (None where not needed) from dout, differentiable themselves."""
    g = iter(torch.autograd.grad(out, [t for t, n in zip(inputs, need) if n], dout, create_graph=True))
    return [next(g) if n else None for n in need]


def _scan_setup(ctx, inputs, output):
    A, B, Wi, Wf, Wr, bi, bf, br, mask, V0, num_heads, n_lv = inputs
    _, pre, states = output
    ctx.set_materialize_grads(False)
    ctx.save_for_backward(A, B, Wi, Wf, Wr, bi, bf, br, mask, V0, pre, states)
    ctx.sizes = (num_heads, n_lv)
    ctx.dtypes = [t.dtype for t in (A, B, Wi, Wf, Wr, bi, bf, br)]


def _scan_backward(ctx, grads):
    dV = grads[0]
    if dV is None:
        return (None,) * 12
    A, B, Wi, Wf, Wr, bi, bf, br, mask, V0, pre, states = ctx.saved_tensors
    if torch.is_grad_enabled():                                                # create_graph: gradients of these are wanted
        ins = [t.view_as(t) for t in (A, B, Wi, Wf, Wr, bi, bf, br, V0)]
        g = _grads_again(_scan_again(*ins, mask, *ctx.sizes), ins, [ctx.needs_input_grad[i] for i in (*range(8), 9)], dV)
        return (*g[:8], None, g[8], None, None)
    wide = any(dt != A.dtype for dt in ctx.dtypes)
    dV0, *rest = torch.ops.dispatcher.gate_scan_train_bwd(A, B, Wi, Wf, Wr, mask, V0, pre, states, dV, *ctx.sizes, wide)
    return (*[g.to(dt) for g, dt in zip(rest, ctx.dtypes)], None, dV0, None, None)


torch.library.register_autograd("dispatcher::gate_scan_train", _scan_backward, setup_context=_scan_setup)


def gate_scan_train(A, B, Wi, Wf, Wr, bi, bf, br, n_lv, mask, V0, num_heads):
    """Scanned mixer state (b, T, d) as fused_gate_scan's, differentiable in everything but the mask: fused_gate_preacts
    and the level loop of the eager mixer (reference dispatcher_hybrid/modeling_dispatcher.py:100-121). Sums and the states
    within a launch are fp32; the pre-activations, the state entering every level and their gradients are kept in A's dtype.
    `mask`: the (T, L) level mask or the (b, T, L) document mask; edges with t < 2^l do not exist whatever it says. See
    scan_fits."""
    return torch.ops.dispatcher.gate_scan_train(A, B, Wi, Wf, Wr, bi, bf, br, mask, V0, num_heads, n_lv)[0]


# ---------------------------------------------------------------------------------------------
# products of a training pass
# ---------------------------------------------------------------------------------------------
def _linear(x2, w, max_rows):
    """x2 (M, K) . w^T: dh_proj_gemm in bf16 up to max_rows rows (measured in fused_gates), else the library."""
    if x2.dtype == torch.bfloat16 and x2.shape[0] <= max_rows and w.shape[1] % 64 == 0 and w.shape[0] % 4 == 0:
        return projections_launch(x2, [w])[0]
    return F.linear(x2, w)


def weight_grads(pairs):
    """[dY^T X for X (M, K), dY (M, N) in pairs], up to four over the same M rows: bf16 as one dh_wgrad_gemm (fp32 sums in a
    fixed order, rounded once), fp32 by the library. Rows with unit stride, 16-byte aligned."""
    if pairs[0][0].dtype != torch.bfloat16:
        return [torch.mm(dy.t(), x) for x, dy in pairs]
    n, M, dev = len(pairs), pairs[0][0].shape[0], pairs[0][0].device
    outs = [torch.empty(dy.shape[1], x.shape[1], device=dev, dtype=x.dtype) for x, dy in pairs]
    vps, i64s, i32s = ctypes.c_void_p * n, ctypes.c_int64 * n, ctypes.c_int * n
    K, N = i32s(*[x.shape[1] for x, _ in pairs]), i32s(*[dy.shape[1] for _, dy in pairs])
    nbytes = _hip.lib.dh_wgrad_gemm_workspace_bytes(M, n, N, K)
    ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=dev)
    st = _hip.lib.dh_wgrad_gemm(
        _hip.DH_BF16, M, n, vps(*[x.data_ptr() for x, _ in pairs]), i64s(*[x.stride(0) for x, _ in pairs]), K,
        vps(*[dy.data_ptr() for _, dy in pairs]), i64s(*[dy.stride(0) for _, dy in pairs]), N,
        vps(*[o.data_ptr() for o in outs]), _hip.ptr(ws), ws.numel(), _hip.stream_handle(dev))
    _hip.check(st, "dh_wgrad_gemm")
    return outs


# fp32 products over few rows go layer by layer: the library splits the terms of a single layer's product there, and its
# concatenated or batched form sums them in one chain, further from exact (input gradient at d = 1024, up to 128 rows:
# 2.9e-7 against 5.7e-7; from 192 rows on, and at d = 512, the two are equal).
SEPARATE_F32_MAX_ROWS = 256


def _separate(x2):
    return x2.dtype == torch.float32 and x2.shape[0] <= SEPARATE_F32_MAX_ROWS


def _input_projections(x2, W, W_cat):
    """Rows [x . w^T for w in W] of the three input projections (W_cat: W concatenated)."""
    if _separate(x2):
        return torch.cat([F.linear(x2, w) for w in W], 1)
    return _linear(x2, W_cat, PROJ_GEMM_MAX_ROWS)


def _input_grad(dproj, W_cat):
    """dproj (M, 3 d) . W_cat (3 d, d), the input's gradient from three projections. bf16: one product (fp32 sums, rounded
    once). fp32: three products over d terms each, added (one fp32 sum over 3 d terms is further from exact: 9.9e-7 against
    5.7e-7 at d = 1024); batched into one call where the rows allow it (25 us of host time against 58)."""
    if dproj.dtype == torch.bfloat16:
        return torch.mm(dproj, W_cat)
    M, d = dproj.shape[0], W_cat.shape[1]
    if not _separate(dproj):
        return torch.bmm(dproj.view(M, 3, d).transpose(0, 1), W_cat.view(3, d, d)).sum(0)
    (a, b, c), W = dproj.split(d, -1), W_cat.split(d)
    return torch.mm(a, W[0]).add_(torch.mm(b, W[1])).add_(torch.mm(c, W[2]))


# ---------------------------------------------------------------------------------------------
# a whole mixer layer
# ---------------------------------------------------------------------------------------------
def mixer_fits(mixer, x, mask, n_lv):
    """The weights mixer_train takes (plain_mixer_weights) if it takes this layer and input, else None: one dtype (fp32 or
    bf16) and device throughout and no autocast, plain bias-free projections, the training scan's limits, and plain eager
    execution (a compiler gets the layer-by-layer form, whose gate path is one registered operation, and a torch.func
    transform that operation's refusal)."""
    if not plain_eager():
        return None
    d, H, dt = mixer.embed_dim, mixer.num_heads, x.dtype
    if not (x.dim() == 3 and type(x) in (torch.Tensor, nn.Parameter) and x.numel() > 0
            and dt in (torch.float32, torch.bfloat16) and x.shape[-1] == d
            and not torch.is_autocast_enabled("cuda") and d == SCAN_HEAD * H and H <= 64 and x.shape[1] <= SCAN_MAX_LEN
            and n_lv <= SCAN_MAX_LEVELS and not mask.requires_grad and mask.device == x.device
            and x.numel() * 3 * x.element_size() < 2 ** 31):                   # 32-bit offsets within the (rows, 3 d) buffers
        return None
    return plain_mixer_weights(mixer, dt, x.device)


class _MixerTrain(torch.autograd.Function):
    """A mixer layer; see mixer_train. An autograd function rather than a registered
    operation: the latter's per-call bookkeeping is ~150 us of host time a direction, as much as a small layer's kernels."""

    @staticmethod
    def forward(ctx, x, W_in, W_x, W_s, Wi, Wf, Wr, bi, bf, br, W_out, mask, num_heads, n_lv):
        b, T, d = x.shape
        x2 = _rows16(x.reshape(b * T, d), 8)
        W_cat = torch.cat((W_in, W_x, W_s))
        proj = _input_projections(x2, (W_in, W_x, W_s), W_cat)                 # rows [V0 | A | B]
        V0, A, B = proj.view(b, T, 3 * d).split(d, -1)
        V, pre, states = _gate_scan_fwd(A, B, (Wi, Wf, Wr), (bi, bf, br), mask, V0, num_heads, n_lv, "mixer_train")
        y = _linear(V.view(b * T, d), W_out, OUT_GEMM_MAX_ROWS)
        ctx.save_for_backward(x, W_in, W_x, W_s, Wi, Wf, Wr, bi, bf, br, W_out, mask, proj, V, pre, states, W_cat)
        ctx.sizes = (num_heads, n_lv)
        return y.view(b, T, d)

    @staticmethod
    def backward(ctx, dy):
        *inputs, mask, proj, V, pre, states, W_cat = ctx.saved_tensors
        num_heads, n_lv = ctx.sizes
        need = ctx.needs_input_grad
        if torch.is_grad_enabled():                                            # create_graph: gradients of these are wanted
            inputs = [t.view_as(t) for t in inputs]                            # (tied weights: a gradient for each use)
            x, W_in, W_x, W_s, *gates, W_out = inputs
            V0, A, B = (F.linear(x, w) for w in (W_in, W_x, W_s))
            y = F.linear(_scan_again(A, B, *gates, V0, mask, num_heads, n_lv), W_out)
            return (*_grads_again(y, inputs, need[:11], dy), None, None, None)
        x, _, _, _, Wi, Wf, Wr, _, _, _, W_out = inputs
        proj, V, W_cat = _dense(proj), _dense(V), _dense(W_cat)
        b, T, d = x.shape
        x2, dy2 = _rows16(x.reshape(b * T, d), 8), _rows16(dy.reshape(b * T, d), 8)
        dV = torch.mm(dy2, W_out).view(b, T, d)
        dproj = torch.empty_like(proj)                                         # rows [dV0 | dA | dB]
        V0, A, B = proj.view(b, T, 3 * d).split(d, -1)
        dV0, dA, dB = dproj.view(b, T, 3 * d).split(d, -1)
        gates = _gate_grads(Wi, d, x.dtype, x.device)
        _gate_scan_bwd(A, B, (Wi, Wf, Wr), mask, V0, pre, states, dV, dV0, [dA, dB] + gates, num_heads, n_lv, "mixer_train")
        dx = _input_grad(dproj, W_cat).view(b, T, d) if need[0] else None
        dw = [None] * 4
        if any(need[i] for i in (1, 2, 3, 10)):
            dw = weight_grads([(x2, g) for g in dproj.split(d, -1)] + [(V.view(b * T, d), dy2)])
        g = [dx, *dw[:3], *gates, dw[3]]
        return (*[v if n else None for v, n in zip(g, need)], None, None, None)


def mixer_train(mixer, x, mask, n_lv, weights):
    """A DispatcherMixer's output (b, T, d), differentiable in x and every parameter (reference
    dispatcher_hybrid/modeling_dispatcher.py:63-123; under create_graph layer by layer, see _scan_again): one product for
    the three input projections, the gate path of gate_scan_train, the output projection; one backward, in which the four
    weight gradients are one launch. `weights` as mixer_fits returns them."""
    ((Wi, bi), (Wf, bf), (Wr, br)), (W_in, W_x, W_s, W_out) = weights
    return _MixerTrain.apply(x, W_in, W_x, W_s, Wi, Wf, Wr, bi, bf, br, W_out, mask, mixer.num_heads, n_lv)


# ---------------------------------------------------------------------------------------------
# a whole attention layer
# ---------------------------------------------------------------------------------------------
def attention_fits(attn, x):
    """The weights (q, k, v, out) attention_train takes if it takes this layer and input, else None: bf16 and one device
    throughout and no autocast, 64-wide heads, plain bias-free projections, plain eager execution."""
    if not plain_eager():
        return None
    d = attn.embed_dim
    if not (x.dim() == 3 and x.is_cuda and type(x) in (torch.Tensor, nn.Parameter) and x.numel() > 0
            and x.dtype == torch.bfloat16 and x.shape[-1] == d and attn.head_dim == 64
            and not torch.is_autocast_enabled("cuda") and x.numel() * 3 * x.element_size() < 2 ** 31):
        return None
    return plain_square_weights((attn.linear_q, attn.linear_k, attn.linear_v, attn.linear_out), d, x.dtype, x.device)


def _attention_grads(inputs, need, dout, cos, sin, H, window):
    """The gradients of an attention layer's (x, W_q, W_k, W_v, W_out) as torch operations that autograd can differentiate
    again; in fp32 (a batched bf16 product with a transposed operand is not used)."""
    from .modeling_dispatcher import causal_window_attention, rope_rotate
    inputs = [t.view_as(t) for t in inputs]                                    # (tied weights: a gradient for each use)
    x, *W = (t.float() for t in inputs)
    b, T, d = x.shape
    q, k, v = (F.linear(x, w).view(b, T, H, d // H).transpose(1, 2) for w in W[:3])
    q, k = (rope_rotate(t, cos.float(), sin.float()) for t in (q, k))
    y = causal_window_attention(q, k, v, window).transpose(1, 2).reshape(b, T, d)
    out = F.linear(y, W[3]).to(inputs[0].dtype)
    return _grads_again(out, inputs, need[:5], dout)


class _AttentionTrain(torch.autograd.Function):
    """An attention layer; see attention_train."""

    @staticmethod
    def forward(ctx, x, W_q, W_k, W_v, W_out, cos, sin, num_heads, window):
        b, T, d = x.shape
        H, hd = num_heads, d // num_heads
        x2 = _rows16(x.reshape(b * T, d), 8)
        W_cat = torch.cat((W_q, W_k, W_v))
        proj = _linear(x2, W_cat, PROJ_GEMM_MAX_ROWS)                          # rows [q | k | v]
        q, k, v = proj.view(b, T, 3 * d).split(d, -1)
        y = torch.empty(b, T, d, device=x.device, dtype=x.dtype)
        kv = torch.empty(2, b, H, T, hd, device=x.device, dtype=x.dtype)       # rotated keys, values, head-major
        lse = torch.empty(b, H, T, device=x.device, dtype=torch.float32)
        p = _hip.ptr
        st = _hip.lib.dh_window_attention_train_fwd(
            _hip.dtype_code(x.dtype), p(q), p(k), p(v), q.stride(0), q.stride(1), p(cos), p(sin), p(y), y.stride(0),
            y.stride(1), p(kv[0]), p(kv[1]), p(lse), b, T, H, hd, window, _hip.stream_handle(x.device))
        _hip.check(st, "attention_train")
        out = _linear(y.view(b * T, d), W_out, OUT_GEMM_MAX_ROWS)
        ctx.save_for_backward(x, W_q, W_k, W_v, W_out, cos, sin, proj, y, kv, lse, W_cat)
        ctx.sizes = (num_heads, window)
        return out.view(b, T, d)

    @staticmethod
    def backward(ctx, dout):
        x, W_q, W_k, W_v, W_out, cos, sin, proj, y, kv, lse, W_cat = ctx.saved_tensors
        H, window = ctx.sizes
        need = ctx.needs_input_grad
        if torch.is_grad_enabled():                                            # create_graph: gradients of these are wanted
            g = _attention_grads((x, W_q, W_k, W_v, W_out), need, dout, cos, sin, H, window)
            return (*g, None, None, None, None)
        cos, sin, proj, y, kv, lse, W_cat = (_dense(t) for t in (cos, sin, proj, y, kv, lse, W_cat))
        b, T, d = x.shape
        hd = d // H
        x2, do2 = _rows16(x.reshape(b * T, d), 8), _rows16(dout.reshape(b * T, d), 8)
        dy = torch.mm(do2, W_out).view(b, T, d)
        dproj = torch.empty_like(proj)                                         # rows [dq | dk | dv]
        q = proj.view(b, T, 3 * d)[..., :d]
        dq, dk, dv = dproj.view(b, T, 3 * d).split(d, -1)
        q_rot = torch.empty(b, H, T, hd, device=x.device, dtype=x.dtype)
        delta = torch.empty_like(lse)
        p = _hip.ptr
        st = _hip.lib.dh_window_attention_bwd(
            _hip.dtype_code(x.dtype), p(q), q.stride(0), q.stride(1), p(kv[0]), p(kv[1]), p(y), y.stride(0), y.stride(1),
            p(dy), dy.stride(0), dy.stride(1), p(lse), p(cos), p(sin), p(q_rot), p(delta), p(dq), p(dk), p(dv),
            dq.stride(0), dq.stride(1), b, T, H, hd, window, _hip.stream_handle(x.device))
        _hip.check(st, "attention_train")
        dx = torch.mm(dproj, W_cat).view(b, T, d) if need[0] else None
        dw = [None] * 4
        if any(need[1:5]):
            dw = weight_grads([(x2, g) for g in dproj.split(d, -1)] + [(y.view(b * T, d), do2)])
        return (*[v if n else None for v, n in zip([dx, *dw], need)], None, None, None, None)


def attention_train(attn, x, weights):
    """A WindowAttention's output (b, T, d), differentiable in x and the four projections (reference
    dispatcher_hybrid/modeling_dispatcher.py:168-182; under create_graph through torch operations): scores and probabilities
    stay in registers in both directions (``dh_window_attention_train_fwd`` / ``dh_window_attention_bwd``; the softmax's
    log-sum is kept in fp32), one product for q, k, v and one launch for the four weight gradients. `weights` as
    attention_fits returns them."""
    T = x.shape[1]
    cos, sin = attn.rope_tables(T, x.device, x.dtype)
    return _AttentionTrain.apply(x, *weights, cos, sin, attn.num_heads, attn.band(T))
