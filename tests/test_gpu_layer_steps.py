"""The routed layer's own launches (sort in blocks, quantisation while gathering, SwiGLU with quantisation, bf16 expert rows)
against the layer as separate library calls: the same kernels for the products, the same roundings - the same bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _layer(fmt, act, H, I, E, k, group, seed):
    import deepseekternarized_amd as bp
    from deepseekternarized_amd.moe import TernaryMoE

    gen = torch.Generator(device="cuda").manual_seed(seed)

    def stack(N, K):
        packed = torch.stack([bp.pack(torch.randint(-1, 2, (N, K), dtype=torch.int8, device="cuda", generator=gen), fmt) for _ in range(min(E, 8))])
        return [(packed[torch.arange(E) % len(packed)].contiguous(), (0.02 * torch.rand(E, N, -(-K // group), device="cuda", generator=gen)).half())]

    return TernaryMoE(stack(I, H), stack(I, H), stack(H, I), H, I, k, fmt, group, act=act), gen


# 4096 ids and more sort in blocks of 1024: whole blocks, a last block of one id, experts without rows, the largest E; matrices
# of 256 columns run on the general kernel
@pytest.mark.parametrize("T,E,k", [(1024, 64, 4), (4097, 8, 1), (700, 512, 8), (820, 384, 6)])
@pytest.mark.parametrize("skew", [0.0, 4.0])
def test_sort_in_blocks(T, E, k, skew):
    moe, gen = _layer("tq2", "bf16", 256, 256, E, k, 64, 20)
    x = torch.randn(T, 256, device="cuda", generator=gen).bfloat16()
    logits = torch.randn(T, E, device="cuda", generator=gen) - skew * torch.arange(E, device="cuda") / E
    assert torch.equal(moe(x, logits), moe.composed(x, logits))


# rows of 1, 2 and 4 pieces per thread in either kernel, and lengths past them (9216: the launches of their own); the decode
# kernels, the 16-token kernel and the general one
@pytest.mark.parametrize("T", [1, 3, 40, 64])
@pytest.mark.parametrize("fmt,H,I,group", [("tq2", 1024, 1024, 128), ("tq1", 2304, 1280, 128), ("tq2", 4352, 2304, 128), ("tq2", 328, 200, 64), ("tq2", 1024, 4608, 128), ("tq2", 9216, 1024, 128)])
def test_int8_rows_are_quantised_where_they_are_made(T, fmt, H, I, group):
    moe, gen = _layer(fmt, "int8", H, I, 8, 2, group, 21)
    x = torch.randn(T, H, device="cuda", generator=gen).bfloat16()
    x[0, :] = 0
    logits = torch.randn(T, 8, device="cuda", generator=gen)
    assert torch.equal(moe(x, logits), moe.composed(x, logits))
