"""Decode launches with many fewer token rows than experts, whose grid holds one y per row (the j-th expert with rows) instead of
one per expert: every expert that has rows must be found, wherever it is."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# one row in the first / last expert and across the scan's blocks of 64 and 256 experts; experts with several rows (fewer
# experts than grid rows); exactly an eighth as many rows as experts, and one more (one y per expert again)
@pytest.mark.parametrize("E,rows", [(64, {0: 1}), (64, {63: 1}), (64, {5: 2, 40: 3}), (130, {63: 1, 64: 1, 127: 1, 128: 1, 129: 1}), (300, {255: 1, 256: 2, 299: 4}),
                                    (600, {511: 1, 512: 1, 599: 9}), (24, {3: 2, 23: 1}), (24, {3: 2, 22: 1, 23: 1})])
@pytest.mark.parametrize("fmt", ["tq1", "tq2"])
@pytest.mark.parametrize("act", ["bf16", "int8", "f32"])
def test_experts_with_rows_are_found(E, rows, fmt, act):
    import deepseekternarized_amd as bp

    N, K = 80, 1024
    gen = torch.Generator(device="cuda").manual_seed(E)
    packed = bp.pack(torch.randint(-1, 2, (E * N, K), dtype=torch.int8, device="cuda", generator=gen), fmt).view(E, N, -1)
    scale = (0.02 * torch.rand(E, N, K // 128, device="cuda", generator=gen)).half()
    counts = [rows.get(e, 0) for e in range(E)]
    T = sum(counts)
    offsets = torch.tensor([0] + counts, dtype=torch.int64).cumsum(0).cuda()
    if act == "int8":
        x, xs = torch.randint(-127, 128, (T, K), dtype=torch.int8, device="cuda", generator=gen), torch.rand(T, device="cuda", generator=gen)
    else:
        x, xs = torch.randn(T, K, device="cuda", generator=gen).to(torch.float32 if act == "f32" else torch.bfloat16), None
    got = bp.grouped_ternary_gemm(x, xs, offsets, packed, scale, K, 128, fmt, max_rows=max(counts))
    ref = bp.grouped_ternary_gemm(x, xs, offsets, packed, scale, K, 128, fmt, max_rows=max(counts), backend="torch")
    # float32 sums of 1024 products in another order, activations to 2^-17 of their block's largest magnitude
    assert float((got.double() - ref.double()).norm(dim=1).div(ref.double().norm(dim=1)).max()) <= 4e-5
