"""Gate readouts of short launches. bf16 launches of at most one (tile, level) per CU run the one-shot kernel: the same
products in the same order as the chunked kernel longer launches run, so a row's outputs are the same bits whether it is
alone or one of many. fp32 splits K over two or four wave groups there: against float64, 1024 products in any order stay
within 1024 x 2^-24 of the sum of their magnitudes; 2e-5 of the largest output is that bound at these magnitudes."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(b, T, GH, H, L, dtype):
    g = torch.Generator(device=DEV).manual_seed(T + GH)
    rn = lambda *s: torch.randn(*s, device=DEV, generator=g)
    A, B = rn(b, T, GH).to(dtype), rn(b, T, GH).to(dtype)
    W = [(rn(L, H, GH) * 0.05).to(dtype) for _ in range(3)]
    bias = [rn(L, H).to(dtype) for _ in range(3)]
    mask = (torch.rand(b, T, L, device=DEV, generator=g) < 0.8).to(dtype)
    return A, B, W, bias, mask


@pytest.mark.parametrize("GH", [256, 512, 768, 1024])
@pytest.mark.parametrize("T,H", [(1, 16), (63, 5), (64, 16), (65, 1), (200, 16)])
def test_one_shot_readouts_equal_the_chunked_kernel(T, H, GH):
    from dispatcher_hybrid.fused_gates import fused_gate_preacts
    n_lv = min(8, T.bit_length())
    A, B, W, bias, mask = _inputs(1, T, GH, H, 8, torch.bfloat16)
    many = 1 + 256 // (((T + 63) // 64) * n_lv)                       # past one workgroup per CU
    for m in (None, mask[..., :n_lv]):
        alone = fused_gate_preacts(A, B, *W, *bias, n_lv, m)
        rep = lambda t: None if t is None else t.expand(many, -1, -1).contiguous()
        batch = fused_gate_preacts(rep(A), rep(B), *W, *bias, n_lv, rep(m))
        for x, y in zip(alone, batch):
            assert torch.equal(x.expand_as(y), y)


@pytest.mark.parametrize("T", [1, 64, 200, 1100, 1700])               # four groups up to 256 workgroups, two up to 448, one
def test_fp32_readouts_with_split_k(T):
    from dispatcher_hybrid.fused_gates import fused_gate_preacts
    n_lv = min(12, T.bit_length())
    A, B, W, bias, mask = _inputs(1, T, 1024, 16, 12, torch.float32)
    got = fused_gate_preacts(A, B, *W, *bias, n_lv, mask[..., :n_lv])
    for l in range(n_lv):
        lag = 1 << l
        src = torch.zeros_like(B, dtype=torch.float64)
        if lag < T:
            src[:, lag:] = B[:, :T - lag].double()
        hid = torch.relu(A.double() + src * (mask[..., l:l + 1] > 0)) ** 2
        for p, w, c in zip(got, W, bias):
            ref = hid @ w[l].double().T + c[l].double()
            assert (p[:, :, l].double() - ref).abs().max() <= 2e-5 * ref.abs().max()
