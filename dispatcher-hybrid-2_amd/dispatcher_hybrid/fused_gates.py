"""Fused gate pipeline of the parallel (prefill / training) forward, on gfx950 HIP kernels.

    model.enable_fused_gates()

Drop-in for the reference module of the same name (reference dispatcher_hybrid/fused_gates.py):
the custom ops ``dispatcher::gate_preacts_fwd`` / ``dispatcher::gate_preacts_bwd`` keep their
schemas (reference :186-190, :225-229), fake implementations and autograd registration, and
``fused_gate_preacts`` keeps its signature (reference :307-314). They compute

    hidden = relu(A + m * roll(B, 2^l))^2            (never materialised)
    pre_x  = hidden . W_x[l] + b_x[l]                x in {i, f, r}

in one kernel (``dh_gate_preacts_fwd``). Dtype rule: bf16 (and fp16) inputs compute in bf16 with
fp32 accumulation and return bf16, like the reference; fp32 inputs compute and return fp32 (the
reference op rounds fp32 models to bf16, which cannot meet a 1e-4 relative tolerance).

Also registered here: ``dispatcher::level_scan_fwd``, the sigmoid/mask/level-scan half of the
mixer (``dh_level_scan_fwd``), which the reference runs as eager torch ops
(reference dispatcher_hybrid/modeling_dispatcher.py:86-88, 111-121).

``silu_mul`` is the feed-forward block's SwiGLU activation in one launch (``dh_silu_mul``);
``add_rmsnorm`` a residual add and the RMSNorm after it (``dh_add_rmsnorm``).

Importing this module loads the kernel library and raises ImportError if it is missing.
"""

import ctypes
from typing import List, Optional

import torch
import torch.nn as nn
from torch.autograd import forward_ad
from torch.nn.modules.module import _has_any_global_hook
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from . import _hip


def _compute_dtype(x):
    return torch.float32 if x.dtype == torch.float32 else torch.bfloat16


def _mask_view(mask, cd, b, T, n_lv):
    """(b, T, >= n_lv) mask in dtype `cd` and its element strides (any layout; no copy if already cd). Sizes that neither
    match nor broadcast raise: the kernels read b x T x n_lv elements by these strides."""
    if mask is None:
        return None, 0, 0, 0
    if mask.dim() != 3:
        raise ValueError(f"document mask: (b, T, levels) expected, got {tuple(mask.shape)}")
    if mask.shape[0] != b or mask.shape[1] != T or mask.shape[2] < n_lv:
        mask = mask[..., :n_lv].expand(b, T, n_lv)
    m = mask.to(cd)
    return m, m.stride(0), m.stride(1), m.stride(2)


def _preacts_launch(A_, B_, Wi_, Wf_, Wr_, bi_, bf_, br_, mask, outs, ostrides, activate, n_lv, what):
    b, T, GH = A_.shape
    H = Wi_.shape[1]
    cd = A_.dtype
    _hip.same_gpu(what, A_, B_, Wi_, Wf_, Wr_, bi_, bf_, br_, mask)
    m_, smb, smt, sml = _mask_view(mask, cd, b, T, n_lv)
    p = _hip.ptr
    st = _hip.lib.dh_gate_preacts_fwd(
        _hip.dtype_code(cd), p(A_), p(B_), A_.stride(0), A_.stride(1),
        p(Wi_), p(Wf_), p(Wr_), Wi_.stride(0), Wi_.stride(1),
        p(bi_), p(bf_), p(br_), p(m_), smb, smt, sml,
        p(outs[0]), p(outs[1]), p(outs[2]), *ostrides, int(activate) | (2 if bi_.dtype == cd else 0),
        b, T, GH, H, n_lv, _hip.stream_handle(A_.device))
    _hip.check(st, what)


def _prep_gate_inputs(A, B, Wi, Wf, Wr, bi, bf, br, n_lv):
    cd = _compute_dtype(A)
    A_, B_ = (_rows16(t.contiguous().to(cd), 8) for t in (A, B))
    Wi_, Wf_, Wr_ = (_rows16(w[:n_lv].contiguous().to(cd), 8) for w in (Wi, Wf, Wr))
    # the kernel reads biases of the compute dtype as they are, others as fp32 copies
    bd = cd if bi.dtype == bf.dtype == br.dtype == cd else torch.float32
    bi_, bf_, br_ = (v[:n_lv].contiguous().to(bd) for v in (bi, bf, br))
    return A_, B_, Wi_, Wf_, Wr_, bi_, bf_, br_


# ---------------------------------------------------------------------------------------------
# dispatcher::gate_preacts_fwd
# ---------------------------------------------------------------------------------------------
@torch.library.custom_op("dispatcher::gate_preacts_fwd", mutates_args=(), device_types="cuda")
def _gate_preacts_fwd_op(A: torch.Tensor, B: torch.Tensor,
                         Wi: torch.Tensor, Wf: torch.Tensor, Wr: torch.Tensor,
                         bi: torch.Tensor, bf: torch.Tensor, br: torch.Tensor,
                         n_lv: int, mask: Optional[torch.Tensor]) -> List[torch.Tensor]:
    b, T, GH = A.shape
    H = Wi.shape[1]
    cd = _compute_dtype(A)
    outs = [torch.empty(b, T, n_lv, H, device=A.device, dtype=cd) for _ in range(3)]
    if b == 0 or T == 0:
        return outs
    ins = _prep_gate_inputs(A, B, Wi, Wf, Wr, bi, bf, br, n_lv)
    o = outs[0]
    _preacts_launch(*ins, mask, outs, (o.stride(0), o.stride(1), o.stride(2), o.stride(3)), 0, n_lv,
                    "dispatcher::gate_preacts_fwd")
    return outs


@_gate_preacts_fwd_op.register_fake
def _(A, B, Wi, Wf, Wr, bi, bf, br, n_lv, mask):
    b, T, _ = A.shape
    H = Wi.shape[1]
    cd = _compute_dtype(A)
    return [A.new_empty(b, T, n_lv, H, dtype=cd) for _ in range(3)]


# ---------------------------------------------------------------------------------------------
# dispatcher::gate_preacts_bwd
# ---------------------------------------------------------------------------------------------
def _rows16(t, n):
    """t with unit-stride rows whose starts are 16-byte aligned (n elements to 16 bytes) and lie at least a row apart; any
    other layout (broadcast or overlapping rows, columns of a wider tensor, an odd offset) copied."""
    w = t.shape[-1]
    if t.stride(-1) == 1 and t.data_ptr() % 16 == 0 and all(s % n == 0 and s >= w for s in t.stride()[:-1]):
        return t
    return t.clone(memory_format=torch.contiguous_format)


def _preacts_bwd_launch(A, B, Wi, Wf, Wr, dP, mask, outs, n_lv, levels, what):
    """dh_gate_preacts_bwd_ws into outs = [dA, dB, dWi, dWf, dWr, dbi, dbf, dbr] (one dtype; dA and dB with unit-stride rows
    and equal strides, the others contiguous with `levels` levels) from dP, three gradients logically (b, T, n_lv, H) with
    one set of strides."""
    b, T, GH = A.shape
    H = Wi.shape[1]
    cd = _compute_dtype(A)
    vec = 8 if cd == torch.bfloat16 else 4
    A_, B_ = (_rows16(t.to(cd), vec) for t in (A, B))
    if A_.stride() != B_.stride():
        A_, B_ = A_.contiguous(), B_.contiguous()
    Wi_, Wf_, Wr_ = (_rows16(w[:n_lv].contiguous().to(cd), vec) for w in (Wi, Wf, Wr))
    if not (dP[0].stride() == dP[1].stride() == dP[2].stride()):
        dP = [g.contiguous() for g in dP]
    _hip.same_gpu(what, A_, B_, Wi_, Wf_, Wr_, *dP, mask)
    m_, smb, smt, sml = _mask_view(mask, cd, b, T, n_lv)
    p = _hip.ptr
    code = _hip.dtype_code(cd)
    nbytes = _hip.lib.dh_gate_preacts_bwd_workspace_bytes(code, b, T, GH, H, n_lv)
    ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=A.device)     # refused sizes: the call below says why
    st = _hip.lib.dh_gate_preacts_bwd_ws(
        code, p(A_), p(B_), A_.stride(0), A_.stride(1), p(Wi_), p(Wf_), p(Wr_), Wi_.stride(0), Wi_.stride(1),
        *[p(g) for g in dP], *dP[0].stride(), p(m_), smb, smt, sml, _hip.dtype_code(outs[0].dtype), p(outs[0]), p(outs[1]),
        outs[0].stride(0), outs[0].stride(1), *[p(o) for o in outs[2:]], levels, b, T, GH, H, n_lv, p(ws), ws.numel(),
        _hip.stream_handle(A.device))
    _hip.check(st, what)


@torch.library.custom_op("dispatcher::gate_preacts_bwd", mutates_args=(), device_types="cuda")
def _gate_preacts_bwd_op(A: torch.Tensor, B: torch.Tensor,
                         Wi: torch.Tensor, Wf: torch.Tensor, Wr: torch.Tensor,
                         dPi: torch.Tensor, dPf: torch.Tensor, dPr: torch.Tensor,
                         n_lv: int, mask: Optional[torch.Tensor]) -> List[torch.Tensor]:
    b, T, GH = A.shape
    H = Wi.shape[1]
    dev = A.device
    f32 = torch.float32
    outs = [torch.empty(b, T, GH, device=dev, dtype=f32), torch.empty(b, T, GH, device=dev, dtype=f32)]
    outs += [torch.empty(n_lv, H, GH, device=dev, dtype=f32) for _ in range(3)]
    outs += [torch.empty(n_lv, H, device=dev, dtype=f32) for _ in range(3)]
    if b == 0 or T == 0:
        for o in outs:
            o.zero_()
        return outs
    cd = _compute_dtype(A)
    _preacts_bwd_launch(A, B, Wi, Wf, Wr, [g.to(cd) for g in (dPi, dPf, dPr)], mask, outs, n_lv, n_lv,
                        "dispatcher::gate_preacts_bwd")
    return outs


@_gate_preacts_bwd_op.register_fake
def _(A, B, Wi, Wf, Wr, dPi, dPf, dPr, n_lv, mask):
    b, T, GH = A.shape
    H = Wi.shape[1]
    f32 = torch.float32
    return ([A.new_empty(b, T, GH, dtype=f32), A.new_empty(b, T, GH, dtype=f32)]
            + [A.new_empty(n_lv, H, GH, dtype=f32) for _ in range(3)]
            + [A.new_empty(n_lv, H, dtype=f32) for _ in range(3)])


def _setup_context(ctx, inputs, output):
    A, B, Wi, Wf, Wr, bi, bf, br, n_lv, mask = inputs
    ctx.save_for_backward(A, B, Wi, Wf, Wr)
    ctx.n_lv = n_lv
    ctx.mask = mask
    ctx.dtypes = (A.dtype, B.dtype, Wi.dtype, bi.dtype)


def _backward(ctx, grads):
    dPi, dPf, dPr = grads
    A, B, Wi, Wf, Wr = ctx.saved_tensors
    n_lv = ctx.n_lv
    z = lambda g: g if g is not None else torch.zeros(
        A.shape[0], A.shape[1], n_lv, Wi.shape[1], device=A.device, dtype=_compute_dtype(A))
    dA, dB, dWi, dWf, dWr, dbi, dbf, dbr = torch.ops.dispatcher.gate_preacts_bwd(
        A, B, Wi, Wf, Wr, z(dPi), z(dPf), z(dPr), n_lv, ctx.mask)
    a_dt, b_dt, w_dt, bias_dt = ctx.dtypes
    levels = Wi.shape[0]

    def pad(g, dt):
        if g.shape[0] == levels:
            return g.to(dt)
        out = torch.zeros((levels,) + tuple(g.shape[1:]), device=g.device, dtype=dt)
        out[:n_lv] = g
        return out

    return (dA.to(a_dt), dB.to(b_dt), pad(dWi, w_dt), pad(dWf, w_dt), pad(dWr, w_dt),
            pad(dbi, bias_dt), pad(dbf, bias_dt), pad(dbr, bias_dt), None, None)


torch.library.register_autograd("dispatcher::gate_preacts_fwd", _backward, setup_context=_setup_context)


def fused_gate_preacts(A, B, Wi, Wf, Wr, bi, bf, br, n_lv, mask=None):
    """(pre_i, pre_f, pre_r), each (b, T, n_lv, H), differentiable and opaque to torch.compile.

    Equal to einsum('btlg,lhg->btlh', relu(A.unsqueeze(2) + m * roll(B, 2^l))**2, W_x[:n_lv]) +
    b_x[:n_lv]; `mask` is the optional (b, T, n_lv) doc-reset mask, the wrap mask t >= 2^l is
    always applied. Same signature as reference dispatcher_hybrid/fused_gates.py:307-314.
    """
    out = torch.ops.dispatcher.gate_preacts_fwd(A, B, Wi, Wf, Wr, bi, bf, br, n_lv, mask)
    return out[0], out[1], out[2]


# ---------------------------------------------------------------------------------------------
# dispatcher::level_scan_fwd
# ---------------------------------------------------------------------------------------------
@torch.library.custom_op("dispatcher::level_scan_fwd", mutates_args=(), device_types="cuda")
def _level_scan_fwd_op(pre_i: torch.Tensor, pre_f: torch.Tensor, pre_r: torch.Tensor,
                       mask: Optional[torch.Tensor], V0: torch.Tensor, num_heads: int,
                       n_lv: int) -> torch.Tensor:
    b, T, d = V0.shape
    out = torch.empty(b, T, d, device=V0.device, dtype=V0.dtype)
    if b == 0 or T == 0:
        return out
    _scan_launch(pre_i, pre_f, pre_r, mask, V0, out, num_heads, n_lv, 0, "dispatcher::level_scan_fwd")
    return out


def _scan_launch(pre_i, pre_f, pre_r, mask, V0, out, num_heads, n_lv, activated, what, ring=None, ring_L=0):
    b, T, d = V0.shape
    cd = V0.dtype
    V0_ = _rows16(V0, 16 // V0.element_size())
    pi, pf, pr = (g.to(cd) for g in (pre_i, pre_f, pre_r))       # keeps each tensor's layout
    if not (pi.stride() == pf.stride() == pr.stride()):
        pi, pf, pr = pi.contiguous(), pf.contiguous(), pr.contiguous()
    _hip.same_gpu(what, V0_, pi, pf, pr, mask)
    m_, smb, smt, sml = _mask_view(mask, cd, b, T, n_lv)
    p = _hip.ptr
    st = _hip.lib.dh_level_scan_fwd(
        _hip.dtype_code(cd), p(pi), p(pf), p(pr), *pi.stride(), p(m_), smb, smt, sml,
        p(V0_), V0_.stride(0), V0_.stride(1), p(out), b, T, num_heads, d // num_heads, n_lv,
        int(activated), p(ring), int(ring_L), _hip.stream_handle(V0.device))
    _hip.check(st, what)


@_level_scan_fwd_op.register_fake
def _(pre_i, pre_f, pre_r, mask, V0, num_heads, n_lv):
    return torch.empty_like(V0)


def fused_level_scan(pre_i, pre_f, pre_r, mask, V0, num_heads, n_lv):
    """Scanned mixer state (b, T, d) from the pre-activations and V0 = linear_in(x) (b, T, d).

    Applies a = sigmoid(pre_i)*M, f = sigmoid(pre_f)*M + (1-M), r = sigmoid(pre_r) and the n_lv
    updates V[t] <- f*V[t] + a*r[t-2^l]*V[t-2^l] (reference dispatcher_hybrid/modeling_dispatcher.py
    :111-121), with M = [t >= 2^l] * mask. The result is in (b, T, H*hd) layout, ready for
    linear_out (no heads-first transposes). Inference only (no autograd).
    """
    return torch.ops.dispatcher.level_scan_fwd(pre_i, pre_f, pre_r, mask, V0, num_heads, n_lv)


# ---------------------------------------------------------------------------------------------
# dispatcher::gate_scan_fwd -- the whole inference gate path in two launches
# ---------------------------------------------------------------------------------------------
def _gate_scan_body(A, B, Wi, Wf, Wr, bi, bf, br, mask, V0, num_heads, n_lv):
    b, T, d = V0.shape
    out = torch.empty(b, T, d, device=V0.device, dtype=V0.dtype)
    if b == 0 or T == 0:
        return out
    ins = _prep_gate_inputs(A, B, Wi, Wf, Wr, bi, bf, br, n_lv)
    H = num_heads
    # activated gates in the head-major (b, H, n_lv, T) layout: unit stride along t for the scan, rows padded to 8
    # positions so they start aligned whatever T is
    g = torch.empty(3, b, H, n_lv, -(-T // 8) * 8, device=V0.device, dtype=ins[0].dtype)
    gates = [x.permute(0, 3, 2, 1)[:, :T] for x in g]                 # logical (b, T, n_lv, H)
    _preacts_launch(*ins, mask, gates, gates[0].stride(), 1, n_lv, "dispatcher::gate_scan_fwd")
    cd = ins[0].dtype
    res = out if V0.dtype == cd else torch.empty(b, T, d, device=V0.device, dtype=cd)
    _scan_launch(gates[0], gates[1], gates[2], None, V0.to(cd), res, H, n_lv, 1, "dispatcher::gate_scan_fwd")
    if res is not out:
        out.copy_(res)
    return out


@torch.library.custom_op("dispatcher::gate_scan_fwd", mutates_args=(), device_types="cuda")
def _gate_scan_fwd_op(A: torch.Tensor, B: torch.Tensor,
                      Wi: torch.Tensor, Wf: torch.Tensor, Wr: torch.Tensor,
                      bi: torch.Tensor, bf: torch.Tensor, br: torch.Tensor,
                      mask: Optional[torch.Tensor], V0: torch.Tensor, num_heads: int,
                      n_lv: int) -> torch.Tensor:
    return _gate_scan_body(A, B, Wi, Wf, Wr, bi, bf, br, mask, V0, num_heads, n_lv)


@_gate_scan_fwd_op.register_fake
def _(A, B, Wi, Wf, Wr, bi, bf, br, mask, V0, num_heads, n_lv):
    return torch.empty_like(V0)


def fused_gate_scan(A, B, Wi, Wf, Wr, bi, bf, br, n_lv, mask, V0, num_heads):
    """Scanned mixer state (b, T, d) straight from the gate hiddens A = gate_hidden(x),
    B = gate_hidden_src(x) and V0 = linear_in(x): the pre-activations are computed, activated and
    masked in one kernel (written head-major, never in the reference op's layout) and the level
    scan consumes them in a second. Inference only (no autograd); equal to
    fused_level_scan(*fused_gate_preacts(...), mask, V0, num_heads, n_lv) up to the bf16 rounding
    of the activated gates, which follows the eager path (reference
    dispatcher_hybrid/modeling_dispatcher.py:86-88, 100-121)."""
    # (wanted gradients go through the registered operation, whose backward says that it has none)
    if type(A) is torch.Tensor and A.is_cuda and plain_eager() and not (torch.is_grad_enabled() and any(
            t.requires_grad for t in (A, B, Wi, Wf, Wr, bi, bf, br, V0))):
        return _gate_scan_body(A, B, Wi, Wf, Wr, bi, bf, br, mask, V0, num_heads, n_lv)
    return torch.ops.dispatcher.gate_scan_fwd(A, B, Wi, Wf, Wr, bi, bf, br, mask, V0, num_heads, n_lv)


def prefill_gate_scan(A, B, Wi, Wf, Wr, bi, bf, br, V0, num_heads, rg_hist, V_ring):
    """Decoder prefill of one tree layer through the parallel kernels: the scanned state (b, T, d)
    plus the decode state the eager prefill fills (reference dispatcher_hybrid/decoding.py:143-185)
    -- rg_hist[:, :T] for every one of the layer's L levels (beyond the prompt's horizon the wrap
    mask is zero, so the transmit gate is sigmoid(relu(A)^2 . W_r + b_r), the eager prefill's
    formula) and, in V_ring, the state entering each level of the last 2^(j+1) positions. Two
    launches: dh_gate_preacts_fwd (activated, all L levels, head-major) and dh_level_scan_fwd over
    the active levels with the ring output; one strided copy moves the transmit gates into
    rg_hist. A, B, V0: (b, T, .) in the state's dtype; no doc-reset mask (a decoder prompt is one
    document)."""
    b, T, d = V0.shape
    L = Wi.shape[0]
    H = num_heads
    cd = _compute_dtype(A)
    if rg_hist.dtype != cd or V_ring.dtype != cd or rg_hist.shape[2] != L:
        raise ValueError("prefill_gate_scan: rg_hist / V_ring must be (b, Tmax, L, H) / (b, S, d) in the compute dtype")
    ins = _prep_gate_inputs(A, B, Wi, Wf, Wr, bi, bf, br, L)
    g = torch.empty(3, b, H, L, T, device=V0.device, dtype=cd)
    gates = [g[i].permute(0, 3, 2, 1) for i in range(3)]              # logical (b, T, L, H)
    _preacts_launch(*ins, None, gates, gates[0].stride(), 1, L, "prefill_gate_scan")
    rg_hist[:, :T].copy_(gates[2])
    n_lv = min(L, T.bit_length())                                       # levels with a source
    out = torch.empty(b, T, d, device=V0.device, dtype=cd)
    _scan_launch(gates[0], gates[1], gates[2], None, V0.to(cd), out, H, n_lv, 1, "prefill_gate_scan",
                 ring=V_ring, ring_L=L)
    return out


def fused_projections(x, weights):
    """[x . W_s^T for W_s in weights] as ONE MFMA GEMM launch (``dh_proj_gemm``) over the
    concatenated weights: the mixer's V0 = linear_in(x), A = gate_hidden(x), B = gate_hidden_src(x)
    (reference dispatcher_hybrid/modeling_dispatcher.py:63-74). x: (..., K) in fp32 or bf16,
    weights: up to three (N_s, K) tensors of x's dtype. Inference only (no autograd)."""
    _hip.require_gpu(x, "fused_projections")
    K = x.shape[-1]
    for w in weights:
        if w.dtype != x.dtype or w.dim() != 2 or w.shape[1] != K or not w.is_contiguous():
            raise ValueError("fused_projections: weights must be contiguous (N, K) tensors of x's dtype")
    _hip.same_gpu("fused_projections", x, *weights)
    return projections_launch(x, weights)


def projections_launch(x, weights):
    """fused_projections of weights that are known to be what it asks for."""
    K = x.shape[-1]
    x2 = _rows16(x.reshape(-1, K), 16 // x.element_size())
    M = x2.shape[0]
    n = len(weights)
    widths = [w.shape[0] for w in weights]
    outs = [torch.empty(*x.shape[:-1], N, device=x.device, dtype=x.dtype) for N in widths]
    if M == 0:
        return outs
    Ws = (ctypes.c_void_p * n)(*[w.data_ptr() for w in weights])
    Ns = (ctypes.c_int * n)(*widths)
    Os = (ctypes.c_void_p * n)(*[o.data_ptr() for o in outs])
    Ls = (ctypes.c_int64 * n)(*widths)
    st = _hip.lib.dh_proj_gemm(_hip.dtype_code(x.dtype), _hip.ptr(x2), x2.stride(0), M, K, n, Ws, Ns, Os, Ls,
                               _hip.stream_handle(x.device))
    _hip.check(st, "dh_proj_gemm")
    return outs


def fitting_weights(x, linears):
    """The layers' weights if dh_proj_gemm gives what calling these layers gives, else None: plain bias-free nn.Linear layers
    (plain_linear), CUDA input, weights of x's dtype, K a multiple of 64 (bf16) / 32 (fp32), output widths multiples of 4."""
    if not (x.is_cuda and len(linears) <= 3 and x.shape[-1] % (64 if x.dtype == torch.bfloat16 else 32) == 0):
        return None
    dt, K, dev = x.dtype, x.shape[-1], x.device
    ws = [plain_weight(l, dt, K, dev) for l in linears]
    return None if any(w is None or w.shape[0] % 4 for w in ws) or _has_any_global_hook() or _function_mode() else ws


def projections_fit(x, linears):
    return fitting_weights(x, linears) is not None


# Rows above which the three library GEMMs (hipBLASLt through nn.Linear) beat dh_proj_gemm for the
# mixer's input projections (measured on MI355X at K = 1024, N = 3 x 1024, bf16, HIP events over 20
# launches: dh_proj_gemm 36 / 61 / 92 / 96 / 190 us against 58 / 63 / 79 / 90 / 173 us for the
# library at M = 4096 / 8192 / 12288 / 16384 / 32768; below 4096 rows dh_proj_gemm takes half the
# library's time or less).
PROJ_GEMM_MAX_ROWS = 8192


def input_projections(x, mixer):
    """V0 = linear_in(x), A = gate_hidden(x), B = gate_hidden_src(x) (reference
    modeling_dispatcher.py:63-74): one dh_proj_gemm launch for a bias-free mixer whose widths the
    kernel takes (K a multiple of 64 for bf16 / 32 for fp32, widths multiples of 4) up to
    PROJ_GEMM_MAX_ROWS rows (the C2 forward and the decoders' prompt prefills); the three nn.Linear
    calls for more rows (the C5 forward's 32768), where the library is faster, and for other layers.
    Inference only."""
    lins = (mixer.linear_in, mixer.gate_hidden, mixer.gate_hidden_src)
    rows = x.numel() // max(x.shape[-1], 1)
    weights = fitting_weights(x, lins) if rows <= PROJ_GEMM_MAX_ROWS else None
    return tuple(l(x) for l in lins) if weights is None else projections_launch(x, weights)


# Rows up to which one dh_proj_gemm launch beats the library, measured on MI355X in captured graphs over 18 distinct weights,
# as in the forward (bf16; us, ours against the library): an attention layer's q, k, v (three 1024-wide nn.Linear GEMMs,
# K = 1024) 21.4 / 32.5 at 2048 rows, 30.2 / 40.0 at 4096, 33.6 / 46.7 at 5120, 44.9 / 51.7 at 6002, 58.2 / 62.9 at 8192; a
# single 1024 x 1024 output projection (the mixer's and attention's linear_out) 6.7 / 8.9 at 1024, 9.3 / 10.7 at 2048,
# 11.4 / 11.5 at 3000, 13.1 / 14.1 at 4096, 15.9 / 14.8 at 4608; the SwiGLU down projection (1024 x 2816) 12.1 / 14.0 at
# 1024, 20.4 / 19.7 at 2048, 25.5 / 22.9 at 3000.
# fp32: the line is a whole mixer layer's, which is one native call up to it (mixer_layer) and separate calls with the
# library's output projection above (eager, us, one call against separate; a call that waits for the host takes ~112): d 512
# 38 / 114 at 24 rows, 49 / 115 at 1024, 69 / 114 at 2048, 100 / 115 at 2750, 104 / 117 at 3012, 118 / 123 at 3500, 127 / 128
# at 4096; d 1024 57 / 114 at 24 rows, 68 / 112 at 200, 106 / 112 at 777, 112 / 112 at 1024, 173 / 171 at 1501, 202 / 195 at
# 2048, 254 / 264 at 2600, 293 / 303 at 3002, 292 / 286 at 3072, 357 / 347 at 4096. Beyond ~1024 rows of d 1024 the two are
# within 4 % either way (the 1024 x 1024 product alone: dh_proj_gemm 24.0 / 33 / 40 / 52 / 58 / 75 us at 1024 / 1501 / 2048 /
# 2500 / 3002 / 4096 rows, the library 19.3 / 32 / 34 / 50 / 68 / 64), so the line stands where d 512 stops gaining much.
QKV_GEMM_MAX_ROWS = 8192
OUT_GEMM_MAX_ROWS = 4096
OUT_GEMM_MAX_ROWS_F32 = 3072
DOWN_GEMM_MAX_ROWS = 1024


# (under autocast the library call casts to the autocast dtype and dh_proj_gemm does not: the line between the two stays at
# half of what the unrestricted bf16 limits are)
def out_max_rows(dtype):
    if torch.is_autocast_enabled("cuda"):
        return OUT_GEMM_MAX_ROWS // 2
    return OUT_GEMM_MAX_ROWS if dtype == torch.bfloat16 else OUT_GEMM_MAX_ROWS_F32


def qkv_max_rows():
    return QKV_GEMM_MAX_ROWS // 2 if torch.is_autocast_enabled("cuda") else QKV_GEMM_MAX_ROWS


def project(x, linears, max_rows):
    """[l(x) for l in linears] (layers over the same input) as one dh_proj_gemm launch when x has at most max_rows rows and
    the kernel takes them (fitting_weights), else the layers' own calls. Inference only."""
    rows = x.numel() // max(x.shape[-1], 1)
    weights = fitting_weights(x, linears) if rows <= max_rows else None
    return [l(x) for l in linears] if weights is None else projections_launch(x, weights)


def _function_mode():
    """Whether a torch-function mode (other than a default device) watches or replaces calls of torch functions."""
    return torch._C._len_torch_function_stack() > 0 and any(
        type(m) is not DeviceContext for m in _get_current_function_mode_stack())


def plain_eager():
    """Whether kernels may be launched without a registered operation around them: no compiler, tracer, torch.func transform
    (grad, vmap, ...), forward-mode level, dispatch mode or function mode looks at the tensors' operations."""
    return not (torch.compiler.is_compiling() or torch._C._are_functorch_transforms_active() or torch.jit.is_tracing()
                or forward_ad._current_level >= 0 or torch._C._len_torch_dispatch_stack() > 0 or _function_mode())


def plain_weight(l, dtype, n_in, device=None):
    """The weight of a bias-free nn.Linear itself (no subclass, adapter, parametrization, replaced forward or hook of its own
    that a direct use of the weight would pass by) if it is a plain contiguous tensor of this dtype and input width, on this
    device if one is given; else None."""
    w = l.weight if type(l) is nn.Linear else None
    if (w is not None and l.bias is None and type(w) in _PLAIN and w.dtype == dtype
            and w.shape[1] == n_in and w.is_contiguous() and w.data_ptr() % 16 == 0 and device in (None, w.device)
            and not (l._forward_hooks or l._forward_pre_hooks or l._backward_hooks or l._backward_pre_hooks
                     or "forward" in l.__dict__)):
        return w
    return None


def plain_linear(l, dtype, n_in, device=None):
    """Whether x . weight^T is all that calling this layer does: plain_weight, no hook on every module and no function mode
    that would see the call of F.linear."""
    return plain_weight(l, dtype, n_in, device) is not None and not _has_any_global_hook() and not _function_mode()


def plain_square_weights(linears, d, dtype, device):
    """The (d, d) weights of these layers if each is plain (plain_linear) and of this dtype and device, else None."""
    ws = [plain_weight(l, dtype, d, device) for l in linears]
    return None if _has_any_global_hook() or _function_mode() or any(w is None or w.shape[0] != d for w in ws) else ws


def plain_mixer_weights(mixer, dtype, device):
    """(gate parameters, projection weights in, x, s, out) of a mixer layer whose (d, d) projections are plain (plain_linear)
    and whose parameters share this dtype and device; else None."""
    gates = mixer._gate_params()
    if not all(w.dtype == dtype and b.dtype == dtype and w.device == device and b.device == device for w, b in gates):
        return None
    lins = plain_square_weights((mixer.linear_in, mixer.gate_hidden, mixer.gate_hidden_src, mixer.linear_out),
                                mixer.embed_dim, dtype, device)
    return None if lins is None else (gates, lins)


_PLAIN = (torch.Tensor, nn.Parameter)


def mixer_layer_fits(mixer, x):
    """The weights mixer_layer takes (plain_mixer_weights) if it takes this layer and input, else None: few enough rows that
    both products run on dh_proj_gemm, one dtype and device throughout, plain bias-free projections, plain eager execution."""
    if not plain_eager():
        return None
    d, dt = mixer.embed_dim, x.dtype
    if not (x.dim() == 3 and type(x) in _PLAIN and dt in (torch.float32, torch.bfloat16) and x.shape[-1] == d
            and 0 < x.shape[0] * x.shape[1] <= out_max_rows(dt) and d % 64 == 0):
        return None
    weights = plain_mixer_weights(mixer, dt, x.device)
    if weights is None or not all(w.is_contiguous() and b.is_contiguous() and w.data_ptr() % 16 == 0 and w.shape[-1] == d
                                  for w, b in weights[0]):
        return None
    return weights


def mixer_layer(mixer, x, mask, n_lv, weights):
    """A DispatcherMixer's output (b, T, d) in one native call (``dh_mixer_fwd``: the launches of fused_projections,
    fused_gate_scan and the output projection, with their results). `mask`: the (b, T, L) document mask, or None; `weights`
    as mixer_layer_fits returns them. Inference only."""
    b, T, d = x.shape
    dt, H = x.dtype, mixer.num_heads
    x2 = _rows16(x.reshape(b * T, d), 8)
    _hip.same_gpu("mixer_layer", x2, mask)
    m, smb, smt, sml = _mask_view(mask, dt, b, T, n_lv)
    code = _hip.dtype_code(dt)
    nbytes = _hip.lib.dh_mixer_fwd_scratch_bytes(code, b, T, d, H, n_lv)
    scratch = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=x.device)
    y = torch.empty(b, T, d, device=x.device, dtype=dt)
    p = _hip.ptr
    ((Wi, bi), (Wf, bf), (Wr, br)), (W_in, W_x, W_s, W_out) = weights
    st = _hip.lib.dh_mixer_fwd(
        code, p(x2), x2.stride(0), p(W_in), p(W_x), p(W_s), p(Wi), p(Wf), p(Wr), p(bi), p(bf), p(br), p(W_out), p(m), smb,
        smt, sml, p(y), p(scratch), scratch.numel(), b, T, d, H, n_lv, _hip.stream_handle(x.device))
    _hip.check(st, "dh_mixer_fwd")
    return y


def swiglu_weights(x, gate, up):
    """The two weights if dh_proj_gemm_swiglu gives silu(gate(x)) * up(x) for these layers, else None: plain bias-free
    nn.Linear layers (plain_linear), a bf16 CUDA input, bf16 weights of one shape, K a multiple of 64 and N of 8."""
    if not (x.is_cuda and x.dtype == torch.bfloat16 and x.shape[-1] % 64 == 0):
        return None
    K, dev = x.shape[-1], x.device
    wg, wu = plain_weight(gate, x.dtype, K, dev), plain_weight(up, x.dtype, K, dev)
    if wg is None or wu is None or wg.shape != wu.shape or wg.shape[0] % 8 or _has_any_global_hook() or _function_mode():
        return None
    return wg, wu


def swiglu_fits(x, gate, up):
    return swiglu_weights(x, gate, up) is not None


def fused_swiglu(x, w_gate, w_up):
    """silu(x . w_gate^T) * (x . w_up^T) as ONE launch (``dh_proj_gemm_swiglu``): the SwiGLU block's
    gate and up GEMMs and its activation (reference dispatcher_hybrid/modeling_dispatcher.py:188-197)
    at the eager rounding points -- both GEMM outputs rounded to bf16, silu rounded, the product
    rounded -- without the two GEMM outputs ever reaching memory. x: (..., K) bf16; w_gate, w_up:
    (N, K) bf16. Returns (..., N). Inference only (no autograd)."""
    _hip.require_gpu(x, "fused_swiglu")
    N, K = w_gate.shape[0], x.shape[-1]
    _hip.same_gpu("fused_swiglu", x, w_gate, w_up)
    if (x.dtype != torch.bfloat16 or w_gate.dtype != torch.bfloat16 or w_up.dtype != torch.bfloat16
            or w_gate.shape != (N, K) or w_up.shape != (N, K) or not w_gate.is_contiguous()
            or not w_up.is_contiguous()):
        raise ValueError("fused_swiglu: bf16 x (..., K) and contiguous bf16 (N, K) gate and up weights")
    return swiglu_launch(x, w_gate, w_up)


def swiglu_launch(x, w_gate, w_up):
    """fused_swiglu of operands that are known to be what it asks for."""
    N, K = w_gate.shape
    x2 = _rows16(x.reshape(-1, K), 8)
    out = torch.empty(*x.shape[:-1], N, device=x.device, dtype=x.dtype)
    M = x2.shape[0]
    if M == 0:
        return out
    st = _hip.lib.dh_proj_gemm_swiglu(_hip.DH_BF16, _hip.ptr(x2), x2.stride(0), M, K, _hip.ptr(w_gate),
                                      _hip.ptr(w_up), N, _hip.ptr(out), N, _hip.stream_handle(x.device))
    _hip.check(st, "dh_proj_gemm_swiglu")
    return out


TREE_MASK_MAX_LEN = 16384
TREE_MASK_MAX_ROWS = 65535
TREE_MASK_MAX_LEVELS = 30


def tree_mask(input_ids, levels, eot, dtype):
    """The parallel forward's tree mask with document resets in ONE launch (``dh_tree_mask``):
    mask[b, t, l] = 1 iff t >= 2^l and no EOT lies among input_ids[b, t-2^l .. t-1], else 0 (the
    level mask times "source and destination in the same document", reference
    dispatcher_hybrid/modeling_dispatcher.py:282-297, 311-323). input_ids: (b, T) int64 CUDA tensor;
    dtype float32 or bfloat16. Returns a contiguous (b, T, levels) tensor of exact 0s and 1s."""
    _hip.require_gpu(input_ids, "tree_mask")
    if input_ids.dim() != 2 or input_ids.dtype != torch.int64 or dtype not in (torch.float32, torch.bfloat16):
        raise ValueError("tree_mask: (b, T) int64 input_ids and a float32 or bfloat16 mask dtype")
    b, T = input_ids.shape
    if not (1 <= levels <= TREE_MASK_MAX_LEVELS) or T > TREE_MASK_MAX_LEN or b > TREE_MASK_MAX_ROWS:
        raise ValueError(f"tree_mask: levels={levels} (1..{TREE_MASK_MAX_LEVELS}), T={T} (<= {TREE_MASK_MAX_LEN}), "
                         f"b={b} (<= {TREE_MASK_MAX_ROWS})")
    # rows of unit stride at least T apart (an expanded batch, stride 0, is copied)
    ids = input_ids if input_ids.stride(1) == 1 and input_ids.stride(0) >= T else input_ids.contiguous()
    out = torch.empty(b, T, levels, device=ids.device, dtype=dtype)
    if b == 0 or T == 0:
        return out
    st = _hip.lib.dh_tree_mask(_hip.dtype_code(dtype), _hip.ptr(ids), ids.stride(0), b, T, levels, int(eot),
                               _hip.ptr(out), _hip.stream_handle(ids.device))
    _hip.check(st, "dh_tree_mask")
    return out


def silu_mul(gate, up, out=None):
    """silu(gate) * up in one launch (``dh_silu_mul``): the SwiGLU activation of reference
    dispatcher_hybrid/modeling_dispatcher.py:197, F.silu(linear_gate(h)) * linear_up(h), at its
    eager rounding points (bf16: silu rounded to bf16, then the product rounded). gate and up:
    same shape, fp32 or bf16 CUDA tensors; out (optional) may be gate or up. Inference only."""
    _hip.require_gpu(gate, "silu_mul")
    if up.shape != gate.shape or up.dtype != gate.dtype or gate.dtype not in (torch.float32, torch.bfloat16):
        raise ValueError("silu_mul: gate and up need one shape and one dtype, fp32 or bf16")
    # contiguous and 16-byte aligned (a view at an odd storage offset is copied)
    g = gate.contiguous() if gate.is_contiguous() and gate.data_ptr() % 16 == 0 else gate.clone()
    u = up.contiguous() if up.is_contiguous() and up.data_ptr() % 16 == 0 else up.clone()
    o = torch.empty_like(g) if out is None else out
    if o.shape != g.shape or o.dtype != g.dtype or not o.is_contiguous():
        raise ValueError("silu_mul: out must be a contiguous tensor of gate's shape and dtype")
    st = _hip.lib.dh_silu_mul(_hip.dtype_code(g.dtype), _hip.ptr(g), _hip.ptr(u), _hip.ptr(o), g.numel(),
                              _hip.stream_handle(g.device))
    _hip.check(st, "dh_silu_mul")
    return o


def _rms_eps(norm):
    # nn.RMSNorm(eps=None) uses the machine epsilon of its fp32 computation type
    return norm.eps if norm.eps is not None else torch.finfo(torch.float32).eps


def add_rmsnorm_fits(d, dtype):
    """Whether dh_add_rmsnorm takes rows of width d in `dtype`: fp32 or bf16, d a multiple of the
    16-byte chunk (8 bf16 or 4 fp32 elements) and at most 64 lanes x 16 chunks of it (8192 bf16,
    4096 fp32 elements)."""
    if dtype not in (torch.float32, torch.bfloat16):
        return False
    v = 8 if dtype == torch.bfloat16 else 4
    return v <= d <= 1024 * v and d % v == 0


def add_rmsnorm(x, y, norm, out=None):
    """(x + y, norm(x + y)) in one launch (``dh_add_rmsnorm``): the residual add of a block and the
    RMSNorm after it (reference dispatcher_hybrid/modeling_dispatcher.py:210-212, 225-227, 341-348).
    x, y: (..., d) fp32 or bf16 CUDA tensors of one shape and dtype; norm: an nn.RMSNorm over d with
    a weight of x's dtype. The sum is written to `out` (x itself may be passed) or a new tensor.
    Inference only."""
    _hip.require_gpu(x, "add_rmsnorm")
    d = x.shape[-1]
    w = norm.weight
    if (y.shape != x.shape or y.dtype != x.dtype or x.dtype not in (torch.float32, torch.bfloat16)
            or w is None or w.dtype != x.dtype or tuple(w.shape) != (d,) or tuple(norm.normalized_shape) != (d,)):
        raise ValueError("add_rmsnorm: x, y need one shape and dtype (fp32 or bf16) and a weighted RMSNorm over "
                         "their last dimension in that dtype")
    xs = x if x.is_contiguous() and x.data_ptr() % 16 == 0 else x.contiguous().clone()
    ys = y if y.is_contiguous() and y.data_ptr() % 16 == 0 else y.contiguous().clone()
    xo = torch.empty_like(xs) if out is None else out
    if xo.shape != x.shape or xo.dtype != x.dtype or not xo.is_contiguous():
        raise ValueError("add_rmsnorm: out must be a contiguous tensor of x's shape and dtype")
    h = torch.empty_like(xs)
    st = _hip.lib.dh_add_rmsnorm(_hip.dtype_code(x.dtype), _hip.ptr(xs), _hip.ptr(ys), _hip.ptr(w),
                                 float(_rms_eps(norm)), _hip.ptr(xo), _hip.ptr(h), xs.numel() // d, d,
                                 _hip.stream_handle(x.device))
    _hip.check(st, "dh_add_rmsnorm")
    return xo, h
