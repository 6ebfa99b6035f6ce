"""``TernaryLinear`` as one library call (``bp_ternary_linear``) against the calls that it stands for: the quantisation, the
grouped product with one expert, the rounding to the output type - the same kernels, so the same bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _weights(fmt, N, K, group, terms, sdt, seed=3):
    import deepseekternarized_amd as bp

    gen = torch.Generator(device="cuda").manual_seed(seed)
    return [bp.PackedTerm(bp.pack(torch.randint(-1, 2, (N, K), dtype=torch.int8, device="cuda", generator=gen), fmt),
                          (0.02 * torch.rand(N, -(-K // group), device="cuda", generator=gen)).to(sdt)) for _ in range(terms)], gen


def _as_tq2(weights, K):
    """What a TQ1 linear of five tokens and more multiplies: the same digits as 2-bit codes."""
    import deepseekternarized_amd as bp

    return [bp.PackedTerm(bp.pack(bp.unpack(w.packed, "tq1", K), "tq2"), w.scale) for w in weights]


def _steps(x, terms, K, group, fmt, act, out_dtype):
    import deepseekternarized_amd as bp
    from deepseekternarized_amd.kernels.ternary_hip import dense_offsets

    q, s = bp.quant_act_int8(x) if act == "int8" else (x, None)
    out = bp.grouped_ternary_gemm(q, s, dense_offsets(x.device, x.size(0)), [t.packed[None] for t in terms], [t.scale[None] for t in terms],
                                  K, group, fmt, max_rows=x.size(0))
    return out.to(out_dtype)


# every decode and small-batch kernel (1 .. 16 rows), a token tile of 32 and its remainder; the general kernel (groups of 64)
@pytest.mark.parametrize("T", [1, 2, 3, 4, 6, 8, 9, 16, 40, 130])
@pytest.mark.parametrize("fmt", ["tq1", "tq2"])
@pytest.mark.parametrize("act,xdt", [("bf16", torch.bfloat16), ("int8", torch.bfloat16), ("bf16", torch.float32), ("int8", torch.float16)])
@pytest.mark.parametrize("N,K,group,terms", [(528, 2048, 128, 1), (2048, 7168, 128, 2), (48, 200, 64, 1)])
def test_linear_call_equals_its_steps(T, fmt, act, xdt, N, K, group, terms):
    import deepseekternarized_amd as bp

    weights, gen = _weights(fmt, N, K, group, terms, torch.float16)
    x = torch.randn(T, K, device="cuda", generator=gen).to(xdt)
    lin = bp.TernaryLinear(weights, K, fmt, group, act=act)
    same, same_fmt = (weights, fmt) if fmt == "tq2" or T < 5 or K % 256 else (_as_tq2(weights, K), "tq2")
    for out_dtype in (torch.bfloat16, torch.float32):
        assert torch.equal(lin(x, out_dtype), _steps(x, same, K, group, same_fmt, act, out_dtype)), out_dtype


def test_weights_that_cannot_be_rewritten_stay_on_their_kernels():
    """TQ1 scales that start 4 bytes into a 16-byte line, which the TQ2 kernels don't read: the TQ1 kernels take the linear as it is, at a size
    that a rewritten one takes to the tiles of 64 - the same exact group sums."""
    import deepseekternarized_amd as bp

    T, N, K = 1100, 4096, 1024
    (w,), gen = _weights("tq1", N, K, 128, 1, torch.float16)
    x = torch.randn(T, K, device="cuda", generator=gen).bfloat16()
    room = torch.empty(w.scale.numel() + 2, dtype=torch.float16, device="cuda")
    scale = room[2:].view(w.scale.shape)
    scale.copy_(w.scale)
    assert scale.data_ptr() % 16 == 4
    want = bp.TernaryLinear([w], K, "tq1", 128)(x, torch.float32)
    assert bp.ext().last_kernel() == "gemm_tq2f4_i8"
    got = bp.TernaryLinear([bp.PackedTerm(w.packed, scale)], K, "tq1", 128)(x, torch.float32)
    assert bp.ext().last_kernel() == "gemm_tq1_i8", bp.ext().last_kernel()
    assert torch.isfinite(got).all() and torch.equal(got, want)


def test_linear_call_with_leading_dimensions():
    import deepseekternarized_amd as bp

    weights, gen = _weights("tq2", 256, 1024, 128, 1, torch.float16)
    lin = bp.TernaryLinear(weights, 1024, "tq2", 128)
    x = torch.randn(2, 3, 1024, device="cuda", generator=gen).bfloat16()
    assert torch.equal(lin(x), lin(x.view(6, 1024)).view(2, 3, 256))


# every digit that a row's 64-code pieces can start at inside a byte, rows at every address modulo 4, one row tile and more rows
# than a workgroup stages, bytes past 242 (which decode to trit 0)
@pytest.mark.parametrize("K", [1024, 1280, 1536, 1792, 2048, 7168])
@pytest.mark.parametrize("N,offset", [(16, 0), (48, 1), (2064, 2), (1024, 3)])
def test_tq1_rows_rewritten_as_tq2(K, N, offset):
    import deepseekternarized_amd as bp

    gen = torch.Generator(device="cuda").manual_seed(K + N)
    Kp = bp.packed_cols("tq1", K)
    bytes_ = torch.randint(0, 256, (N * Kp + offset,), dtype=torch.uint8, device="cuda", generator=gen)
    packed = bytes_[offset:].view(N, Kp)
    weights = [bp.PackedTerm(packed, (0.02 * torch.rand(N, K // 128, device="cuda", generator=gen)).half())]
    x = torch.randn(6, K, device="cuda", generator=gen).bfloat16()
    got = bp.TernaryLinear(weights, K, "tq1", 128, act="bf16")(x, torch.float32)
    assert torch.equal(got, _steps(x, _as_tq2(weights, K), K, 128, "tq2", "bf16", torch.float32))
