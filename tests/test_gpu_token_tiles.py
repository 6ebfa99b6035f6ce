"""How the token-tile kernels deal out their work: launches of one or a few experts, whose (expert, token tile, row block)
triples are split over the XCDs, against the reference-order kernel."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _call(fmt, act, counts, N, K, seed, terms=1, group=128, sdt=torch.float16, max_rows=None, ref=True):
    import deepseekternarized_amd as bp
    from deepseekternarized_amd.ternary.pack import pack

    gen = torch.Generator(device="cuda").manual_seed(seed)
    E, T = len(counts), sum(counts)
    packed, scale = [], []
    for _ in range(terms):
        trits = torch.randint(-1, 2, (E * N, K), dtype=torch.int8, device="cuda", generator=gen)
        packed.append(pack(trits, fmt).view(E, N, -1))
        scale.append((0.01 + 0.02 * torch.rand(E, N, K // group, device="cuda", generator=gen)).to(sdt))
    offsets = torch.tensor([0] + list(counts), dtype=torch.int64).cumsum(0).cuda()
    if act == "int8":
        x = torch.randint(-127, 128, (T, K), dtype=torch.int8, device="cuda", generator=gen)
        xs = 0.01 + 0.02 * torch.rand(T, device="cuda", generator=gen)
    else:
        x, xs = torch.randn(T, K, device="cuda", generator=gen).bfloat16(), None
    args = (x, xs, offsets, packed, scale, K, group, fmt)
    got = bp.grouped_ternary_gemm(*args, max_rows=max_rows or max(counts))
    return got, bp.grouped_ternary_gemm(*args, max_rows=max_rows or max(counts), backend="torch") if ref else None


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


@pytest.fixture
def tune(monkeypatch):
    from deepseekternarized_amd.kernels import _lib

    def set_(name, value):
        monkeypatch.setenv(name, value)
        _lib.load().bp_reload_tuning()

    yield set_
    monkeypatch.undo()
    _lib.load().bp_reload_tuning()


# token tiles of 64: full ones and a remainder of 1, 2, 16, 17, 44 or 63 rows, experts without rows; K of an odd number of
# 256-wide windows and of one scale per 256; 16 rows past a whole row block of 256
@pytest.mark.parametrize("counts", [(130,), (129, 0, 63), (192, 65, 127, 128), (16, 17, 300)])
@pytest.mark.parametrize("N,K,group,terms,sdt", [(256, 1024, 128, 1, torch.float16), (272, 1280, 128, 2, torch.bfloat16), (528, 2048, 256, 1, torch.float32)])
def test_int8_tiles_of_64(tune, counts, N, K, group, terms, sdt):
    import deepseekternarized_amd as bp

    tune("BP_TUNE_TQ2G", "f")
    got, ref = _call("tq2", "int8", counts, N, K, 6, terms, group, sdt, max_rows=300)
    _close(got, ref, "int8")
    _call("tq2", "int8", counts, N, K, 6, terms, group, sdt, max_rows=300, ref=False)
    assert bp.ext().last_kernel() == "gemm_tq2f4_i8"


# longer rows and more terms, an odd number of windows, one scale per 256, remainders of 1 and 63 rows
@pytest.mark.parametrize("counts", [(129, 0, 63), (193, 65, 255)])
@pytest.mark.parametrize("N,K,group,terms,sdt", [(272, 3584, 128, 1, torch.float16), (528, 4352, 128, 1, torch.float32), (256, 2048, 128, 2, torch.bfloat16),
                                                 (272, 2304, 128, 2, torch.float16), (528, 4096, 256, 1, torch.float16), (272, 1280, 128, 3, torch.float32)])
def test_int8_tiles_of_64_with_long_rows_and_terms(tune, counts, N, K, group, terms, sdt):
    import deepseekternarized_amd as bp

    tune("BP_TUNE_TQ2G", "f")
    got, _ = _call("tq2", "int8", counts, N, K, 13, terms, group, sdt, max_rows=300, ref=False)
    assert bp.ext().last_kernel() == "gemm_tq2f4_i8"
    _, ref = _call("tq2", "int8", counts, N, K, 13, terms, group, sdt, max_rows=300)  # (the reference-order kernel's)
    _close(got, ref, "int8")


@pytest.mark.parametrize("T,K,scale", [(129, 1024, 1.0), (200, 1280, 1e-6), (130, 4352, 100.0)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_linear_quantises_in_the_conversion_pass(tune, T, K, scale, out_dtype):
    """The same int8 rows and scales as bp_quant_act_int8 (also for a row of zeros and one with a NaN, and for more groups than
    stay in registers), so the same product as the two calls one after the other."""
    import deepseekternarized_amd as bp
    from deepseekternarized_amd.kernels.ternary_hip import dense_offsets

    gen = torch.Generator(device="cuda").manual_seed(9)
    N = 272
    packed = bp.pack(torch.randint(-1, 2, (N, K), dtype=torch.int8, device="cuda", generator=gen), "tq2")
    s = (0.01 + 0.02 * torch.rand(N, K // 128, device="cuda", generator=gen)).half()
    x = scale * torch.randn(T, K, device="cuda", generator=gen)
    x[3] = 0
    x[5, 7] = float("nan")
    x = x.bfloat16()
    tune("BP_TUNE_TQ2G", "f")
    got = bp.TernaryLinear([bp.PackedTerm(packed, s)], K, "tq2", 128)(x, out_dtype)
    assert bp.ext().last_kernel() == "gemm_tq2f4_i8"
    q, qs = bp.quant_act_int8(x)
    ref = bp.grouped_ternary_gemm(q, qs, dense_offsets(x.device, T), [packed[None]], [s[None]], K, 128, "tq2", max_rows=T).to(out_dtype)
    assert torch.equal(got.isnan(), ref.isnan()) and bool(ref[5].isnan().all())
    assert torch.equal(got.nan_to_num(), ref.nan_to_num())
    # ... and the product itself against the reference-order kernel (both references above run on this kernel)
    ref = bp.grouped_ternary_gemm(q, qs, dense_offsets(x.device, T), [packed[None]], [s[None]], K, 128, "tq2", max_rows=T, backend="torch")
    keep = torch.arange(T, device="cuda") != 5
    bound = 4e-6 if out_dtype == torch.float32 else 2**-9  # (bf16: half a step)
    assert float((got[keep].double() - ref[keep].double()).norm() / ref[keep].double().norm()) <= bound


@pytest.mark.parametrize("pattern,T,E,k,terms,H", [("standard", 1100, 8, 1, 1, 1024), ("standard", 700, 16, 4, 2, 1024), ("v4", 520, 4, 2, 1, 1024),
                                                   ("standard", 1100, 8, 1, 1, 4096), ("standard", 700, 4, 3, 2, 2048), ("v4", 520, 4, 2, 1, 4096)])
def test_int8_layer_on_tiles_of_64(tune, pattern, T, E, k, terms, H):
    """The layer on the 64-token kernel against the same layer as separate launches (standard), or on the 32-token kernel (v4):
    the same rounding points over float32 sums that differ in order, so a few bf16 roundings and int8 steps fall otherwise.
    H = 4096, and 2048 in two terms: long rows in the gate | up launch, which applies SwiGLU and gathers."""
    import deepseekternarized_amd as bp
    from deepseekternarized_amd.moe import TernaryMoE

    gen = torch.Generator(device="cuda").manual_seed(10)
    I = 1280

    def terms_of(N, K):
        return [(torch.stack([bp.pack(torch.randint(-1, 2, (N, K), dtype=torch.int8, device="cuda", generator=gen), "tq2") for _ in range(E)]),
                 (0.02 * torch.rand(E, N, K // 128, device="cuda", generator=gen)).half()) for _ in range(terms)]

    v4 = pattern == "v4"
    moe = TernaryMoE(terms_of(I, H), terms_of(I, H), terms_of(H, I), H, I, k, "tq2", 128, act="int8", pattern=pattern, swiglu_limit=10.0 if v4 else 0.0)
    x = torch.randn(T, H, device="cuda", generator=gen).bfloat16()
    logits = 1.5 * torch.randn(T, E, device="cuda", generator=gen)
    if v4:
        w, idx = torch.topk(torch.softmax(logits, -1), k)
        run = lambda: moe.routed(x, w, idx)  # noqa: E731
    else:
        run = lambda: moe(x, logits)  # noqa: E731
    got = run()
    assert bp.ext().last_kernel() == "gemm_tq2f4_i8+glu+gather+y16"
    if v4:
        tune("BP_TUNE_TQ2G", "b")
        ref = run()
    else:
        ref = moe.composed(x, logits)
    assert torch.isfinite(got).all()
    assert float((got.double() - ref.double()).norm() / ref.double().norm()) <= 4e-3


# few experts with many rows each: 896 to 2048 rows, one and two terms
@pytest.mark.parametrize("T,E,k,I,terms", [(448, 8, 2, 4096, 1), (512, 8, 2, 4096, 1), (1152, 4, 1, 1024, 1), (1280, 4, 1, 1024, 1), (960, 8, 2, 1024, 2), (1024, 8, 2, 1024, 2)])
def test_int8_layers_of_few_experts(T, E, k, I, terms):
    import deepseekternarized_amd as bp
    from deepseekternarized_amd.moe import TernaryMoE

    gen = torch.Generator(device="cuda").manual_seed(11)
    H = 1024

    def terms_of(N, K):
        return [(bp.pack(torch.randint(-1, 2, (E * N, K), dtype=torch.int8, device="cuda", generator=gen), "tq2").view(E, N, -1),
                 (0.02 * torch.rand(E, N, K // 128, device="cuda", generator=gen)).half()) for _ in range(terms)]

    moe = TernaryMoE(terms_of(I, H), terms_of(I, H), terms_of(H, I), H, I, k, "tq2", 128, act="int8")
    x = torch.randn(T, H, device="cuda", generator=gen).bfloat16()
    logits = torch.randn(T, E, device="cuda", generator=gen)
    got = moe(x, logits)
    assert bp.ext().last_kernel() == "gemm_tq2f4_i8+glu+gather+y16"
    ref = moe.composed(x, logits)
    assert float((got.double() - ref.double()).norm() / ref.double().norm()) <= 4e-3  # (bf16 roundings and int8 steps that fall otherwise)


# the rows of tests/test_workspace_sizes.py that lie at a line of the grouped calls', which linears don't have
@pytest.mark.parametrize("T,N,K,terms", [(2048, 2048, 1536, 2), (2048, 2048, 2048, 2), (2048, 2048, 2048, 1), (3072, 2048, 1792, 2), (1536, 4096, 7168, 2)])
def test_int8_linears_on_either_side_of_the_grouped_calls_lines(T, N, K, terms):
    import deepseekternarized_amd as bp

    gen = torch.Generator(device="cuda").manual_seed(12)
    weights = [bp.PackedTerm(bp.pack(torch.randint(-1, 2, (N, K), dtype=torch.int8, device="cuda", generator=gen), "tq2"),
                             (0.02 * torch.rand(N, K // 128, device="cuda", generator=gen)).half()) for _ in range(terms)]
    x = torch.randn(T, K, device="cuda", generator=gen).bfloat16()
    got = bp.TernaryLinear(weights, K, "tq2", 128)(x, torch.float32)
    assert bp.ext().last_kernel() == "gemm_tq2f4_i8"
    ref = bp.TernaryLinear(weights, K, "tq2", 128, backend="torch")(x, torch.float32)
    _close(got, ref, "int8")
