"""dh_gate_preacts_bwd_ws (the matrix-core backward of the gate pre-activations) against a float64 restatement with the
kernel's rounding points: x = relu(a + ok b) and hid = x^2 rounded to the dtype, everything else exact. What remains is
fp32 accumulation: sums of at most N products in any order stay within N 2^-24 of the sum of their magnitudes, and with
random signs far below; 2e-5 of the result's largest value covers the sizes here (N <= 2 * 515 positions or 64 heads x 3
gates x 12 levels)."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _reference(A, B, W, dP, mask, n_lv, dtype):
    b, T, GH = A.shape
    A, B = A.double(), B.double()
    dA, dB = torch.zeros_like(A), torch.zeros_like(A)
    dW = [torch.zeros(w[:n_lv].shape, device=DEV, dtype=torch.float64) for w in W]
    rnd = lambda x: x.to(dtype).double()
    for l in range(n_lv):
        lag = 1 << l
        ok = torch.zeros(b, T, 1, device=DEV, dtype=torch.float64)
        ok[:, lag:] = 1
        if mask is not None:
            ok = ok * (mask[..., l:l + 1] > 0)
        src = torch.zeros_like(B)
        if lag < T:
            src[:, lag:] = B[:, :T - lag]
        x = rnd((A + src * ok).float()).clamp_min(0)
        hid = rnd((x * x).float())
        dh = sum(p[:, :, l].double() @ w[l].double() for p, w in zip(dP, W))
        dx = 2 * x * dh
        dA += dx
        if lag < T:
            dB[:, :T - lag] += (dx * ok)[:, lag:]
        for x_, p in enumerate(dP):
            dW[x_][l] = torch.einsum("bth,btg->hg", p[:, :, l].double(), hid)
    db = [p.double().sum((0, 1)) for p in dP]
    return [dA, dB, *dW, *db]


CASES = [  # b, T, GH, H, n_lv, mask, layout
    (1, 1, 64, 1, 1, False, "op"),
    (2, 15, 64, 5, 4, True, "op"),
    (1, 16, 128, 16, 5, False, "head"),
    (2, 17, 192, 17, 3, True, "head"),
    (1, 33, 64, 8, 6, True, "expanded"),
    (3, 64, 128, 16, 7, True, "op"),
    (2, 130, 1024, 16, 8, True, "head"),
    (1, 515, 256, 64, 10, True, "op"),          # 40 (level, head group) pairs: the weights pass through LDS in chunks
    (1, 5, 64, 2, 3, True, "rows"), (2, 64, 64, 16, 6, True, "rows"), (2, 131, 64, 17, 16, True, "rows"),
    (2, 515, 64, 3, 16, False, "head"),          # levels whose lag exceeds the length
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,T,GH,H,n_lv,masked,layout", CASES)
def test_gate_backward_against_float64(b, T, GH, H, n_lv, masked, layout, dtype):
    from dispatcher_hybrid.fused_gates import _preacts_bwd_launch
    g = torch.Generator(device=DEV).manual_seed(T * 31 + H)
    rn = lambda *s: torch.randn(*s, device=DEV, generator=g)
    A, B = rn(b, T, GH).to(dtype), rn(b, T, GH).to(dtype)
    L = n_lv + 2
    W = [(rn(L, H, GH) * 0.1).to(dtype) for _ in range(3)]
    mask = (torch.rand(b, T, L, device=DEV, generator=g) < 0.8).to(dtype) if masked else None
    if layout == "head":
        dP = [rn(b, H, n_lv, T).to(dtype).permute(0, 3, 2, 1) for _ in range(3)]
    elif layout == "rows":                                        # head-major rows padded to 8, the padding not a number
        dP = [torch.full((b, H, n_lv, -(-T // 8) * 8), float("nan"), device=DEV, dtype=dtype) for _ in range(3)]
        for p in dP:
            p[..., :T] = rn(b, H, n_lv, T).to(dtype)
        dP = [p[..., :T].permute(0, 3, 2, 1) for p in dP]
    elif layout == "expanded":                                    # one value for all positions: stride 0 along t
        dP = [rn(b, 1, n_lv, H).to(dtype).expand(b, T, n_lv, H) for _ in range(3)]
    else:
        dP = [rn(b, T, n_lv, H).to(dtype) for _ in range(3)]
    ref = _reference(A, B, W, dP, mask, n_lv, dtype)

    def run(out_dtype, levels):
        outs = [torch.full((b, T, GH), float("nan"), device=DEV, dtype=out_dtype) for _ in range(2)]
        outs += [torch.full((levels, H, GH), float("nan"), device=DEV, dtype=out_dtype) for _ in range(3)]
        outs += [torch.full((levels, H), float("nan"), device=DEV, dtype=out_dtype) for _ in range(3)]
        _preacts_bwd_launch(A, B, *W, dP, mask, outs, n_lv, levels, "test")
        return outs

    got = run(torch.float32, n_lv)
    for i, (x, y) in enumerate(zip(got, ref)):
        assert (x.double() - y).abs().max() <= 2e-5 * y.abs().max().clamp_min(1e-6), i
    again = run(torch.float32, n_lv)
    assert all(torch.equal(x, y) for x, y in zip(got, again))                 # fixed summation order
    padded = run(dtype, L)                                                   # rounded once, zeros past n_lv
    for x, y in zip(padded[:2], got[:2]):
        assert torch.equal(x, y.to(dtype))
    for x, y in zip(padded[2:], got[2:]):
        assert torch.equal(x[:n_lv], y.to(dtype)) and not x[n_lv:].any()


def test_gate_backward_infinite_source_reaches_only_its_destinations():
    """An infinite source row without a destination leaves every gradient finite: the masked edges contribute nothing."""
    from dispatcher_hybrid.fused_gates import _preacts_bwd_launch
    b, T, GH, H, n_lv = 1, 40, 64, 4, 5
    g = torch.Generator(device=DEV).manual_seed(0)
    A = torch.randn(b, T, GH, device=DEV, generator=g).bfloat16()
    B = torch.randn(b, T, GH, device=DEV, generator=g).bfloat16()
    B[0, 7] = float("inf")
    mask = torch.ones(b, T, n_lv, device=DEV)
    for l in range(n_lv):
        mask[0, 7 + (1 << l), l] = 0
    W = [torch.randn(n_lv, H, GH, device=DEV, generator=g).bfloat16() for _ in range(3)]
    dP = [torch.randn(b, T, n_lv, H, device=DEV, generator=g).bfloat16() for _ in range(3)]
    outs = [torch.empty(b, T, GH, device=DEV) for _ in range(2)]
    outs += [torch.empty(n_lv, H, GH, device=DEV) for _ in range(3)] + [torch.empty(n_lv, H, device=DEV) for _ in range(3)]
    _preacts_bwd_launch(A, B, *W, dP, mask, outs, n_lv, n_lv, "test")
    assert all(bool(o.isfinite().all()) for o in outs) and not outs[1][0, 7].any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,T,GH,H,n_lv,masked", [(1, 1, 64, 1, 1, False), (2, 33, 128, 17, 5, True), (1, 70, 320, 16, 8, True)])
def test_backward_without_scratch_equals_the_one_with(b, T, GH, H, n_lv, masked, dtype):
    """dh_gate_preacts_bwd (the C entry for callers without scratch memory: fp32 atomics, any order) against float64."""
    from dispatcher_hybrid import _hip
    g = torch.Generator(device=DEV).manual_seed(T)
    rn = lambda *s: torch.randn(*s, device=DEV, generator=g).to(dtype)
    A, B, W = rn(b, T, GH), rn(b, T, GH), [rn(n_lv, H, GH) * 0.1 for _ in range(3)]
    dP = [rn(b, T, n_lv, H) for _ in range(3)]
    mask = (torch.rand(b, T, n_lv, device=DEV, generator=g) < 0.8).to(dtype) if masked else None
    outs = [torch.full((b, T, GH), float("nan"), device=DEV) for _ in range(2)]
    outs += [torch.full((n_lv, H, GH), float("nan"), device=DEV) for _ in range(3)]
    outs += [torch.full((n_lv, H), float("nan"), device=DEV) for _ in range(3)]
    p = _hip.ptr
    st = _hip.lib.dh_gate_preacts_bwd(
        _hip.dtype_code(dtype), p(A), p(B), A.stride(0), A.stride(1), *[p(w) for w in W], W[0].stride(0), W[0].stride(1),
        *[p(d) for d in dP], p(mask), *(mask.stride() if masked else (0, 0, 0)), *[p(o) for o in outs], b, T, GH, H, n_lv,
        _hip.stream_handle(A.device))
    _hip.check(st, "dh_gate_preacts_bwd")
    for i, (x, y) in enumerate(zip(outs, _reference(A, B, W, dP, mask, n_lv, dtype))):
        assert (x.double() - y).abs().max() <= 2e-5 * y.abs().max().clamp_min(1e-6), i
