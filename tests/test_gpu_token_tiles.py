"""How the token-tile kernels deal out their work: launches of one or a few experts, whose (expert, token tile, row block)
triples are split over the XCDs, against the reference-order kernel."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _call(fmt, act, counts, N, K, seed, terms=1):
    import deepseekternarized_amd as bp
    from deepseekternarized_amd.ternary.pack import pack

    gen = torch.Generator(device="cuda").manual_seed(seed)
    E, T = len(counts), sum(counts)
    packed, scale = [], []
    for _ in range(terms):
        trits = torch.randint(-1, 2, (E * N, K), dtype=torch.int8, device="cuda", generator=gen)
        packed.append(pack(trits, fmt).view(E, N, -1))
        scale.append((0.01 + 0.02 * torch.rand(E, N, K // 128, device="cuda", generator=gen)).half())
    offsets = torch.tensor([0] + list(counts), dtype=torch.int64).cumsum(0).cuda()
    if act == "int8":
        x = torch.randint(-127, 128, (T, K), dtype=torch.int8, device="cuda", generator=gen)
        xs = 0.01 + 0.02 * torch.rand(T, device="cuda", generator=gen)
    else:
        x, xs = torch.randn(T, K, device="cuda", generator=gen).bfloat16(), None
    args = (x, xs, offsets, packed, scale, K, 128, fmt)
    got = bp.grouped_ternary_gemm(*args, max_rows=max(counts))
    ref = bp.grouped_ternary_gemm(*args, max_rows=max(counts), backend="torch")
    return got, ref


def _close(got, ref, act):
    # int8: the same exact group sums; float32 sums of at most K / 128 * terms = 64 products in other orders: 64 * 2^-24.
    # bf16: two fp8 pieces drop less than 2^-17 of a block's largest magnitude (about 3 standard deviations) per activation.
    bound = 4e-6 if act == "int8" else 4e-5
    assert torch.isfinite(got).all()
    assert float((got.double() - ref.double()).norm() / ref.double().norm()) <= bound


@pytest.mark.parametrize("fmt,act", [("tq1", "bf16"), ("tq1", "int8"), ("tq2", "bf16"), ("tq2", "int8")])
@pytest.mark.parametrize("counts,N", [((129,), 528), ((777,), 512), ((33, 0), 1040), ((65, 1, 200), 272), ((40, 0, 17, 33, 90, 31, 64, 5, 129), 528)])
def test_few_experts(fmt, act, counts, N):
    _close(*_call(fmt, act, counts, N, 1024, 5), act)
