"""dh_wgrad_gemm against float64: each output within half a bf16 spacing of its rounding (at most 2^-8 relative) plus the fp32
accumulation of M products (M 2^-24 of the sum of their magnitudes; 2^-11 of it covers M <= 8192)."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("M,shapes", [
    (1, [(8, 8)]), (63, [(64, 64), (136, 72)]), (64, [(128, 128)]), (65, [(120, 264)]), (511, [(1024, 64)]),
    (1024, [(128, 128), (256, 64), (8, 1000), (512, 136)]),        # split rows, four layers, ragged tiles
    (3001, [(1024, 1024)] * 4), (5000, [(64, 64)]),
    (6143, [(136, 256)]), (6144, [(136, 256), (8, 512)]), (6145, [(1024, 256)]),
    (8001, [(256, 1024)] * 4), (6200, [(64, 264)])])
def test_weight_grads_against_float64(M, shapes):
    from dispatcher_hybrid.fused_train import weight_grads
    g = torch.Generator(device=DEV).manual_seed(M)
    pairs = []
    for N, K in shapes:
        wide = torch.randn(M, N + 24, device=DEV, generator=g).bfloat16()       # a column block of wider rows
        pairs.append((torch.randn(M, K, device=DEV, generator=g).bfloat16(), wide[:, 16:16 + N]))
    got, again = weight_grads(pairs), weight_grads(pairs)
    for (x, dy), w, w2 in zip(pairs, got, again):
        ref = dy.double().t() @ x.double()
        mag = dy.double().abs().t() @ x.double().abs()
        assert w.shape == ref.shape and torch.equal(w, w2)
        assert ((w.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -11 * mag * min(1.0, M / 8192) + 1e-30).all()


def test_weight_grads_propagate_infinity_and_nan():
    from dispatcher_hybrid.fused_train import weight_grads
    x, dy = torch.ones(200, 64, device=DEV).bfloat16(), torch.ones(200, 64, device=DEV).bfloat16()
    x[150, 3], dy[7, 5] = float("inf"), float("nan")
    w = weight_grads([(x, dy)])[0].float()
    assert w[:, 3].isinf().sum() == 63 and w[5].isnan().all()
    keep = torch.ones(64, dtype=torch.bool)
    keep[[3, 5]] = False
    assert (w[[i for i in range(64) if i != 5]][:, [i for i in range(64) if i != 3]] == 200).all()
