"""The GEMM over token tiles of 64: its lines, tiles of at most 32 rows, odd sizes, and what its two pieces of an activation keep."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _terms(E, N, K, terms, gen, sdt=torch.float16, group=128):
    import deepseekternarized_amd as bp

    return [(bp.pack(torch.randint(-1, 2, (E * N, K), dtype=torch.int8, device="cuda", generator=gen), "tq2").view(E, N, -1),
             (0.02 * torch.rand(E, N, -(-K // group), device="cuda", generator=gen)).to(sdt)) for _ in range(terms)]


# int8 layers either side of the lines: 16 rows per expert on average; 128 rows; with 1024 columns 280 tiles of 32 rows x 256 gate | up rows; up to 64
# tokens 384 blocks of 128 columns. Up to 256 routed rows (preparation and tile list in one launch) and more; against the kernels over tiles of 32, whose exact group sums are scaled and added in the same order
@pytest.mark.parametrize("pattern,T,E,k,terms,I,wide", [("standard", 127, 16, 2, 1, 1040, False), ("standard", 128, 16, 2, 1, 1040, True), ("v4", 70, 8, 2, 2, 1280, True),
                                                        ("standard", 333, 16, 3, 2, 1280, True), ("standard", 127, 4, 1, 1, 1280, False), ("standard", 128, 4, 1, 1, 1280, True),
                                                        ("standard", 432, 16, 2, 1, 1024, False), ("v4", 433, 16, 2, 1, 1024, True), ("standard", 64, 47, 12, 1, 1024, False),
                                                        ("standard", 64, 48, 12, 1, 1024, True), ("standard", 64, 8, 4, 2, 1280, False)])
def test_int8_layers_from_sixteen_rows_per_expert(tune, pattern, T, E, k, terms, I, wide):
    import deepseekternarized_amd as bp
    from deepseekternarized_amd.moe import TernaryMoE

    gen = torch.Generator(device="cuda").manual_seed(21)
    H, v4 = 1280, pattern == "v4"
    moe = TernaryMoE(_terms(E, I, H, terms, gen), _terms(E, I, H, terms, gen), _terms(E, H, I, terms, gen), H, I, k, "tq2", 128, act="int8", pattern=pattern,
                     swiglu_limit=10.0 if v4 else 0.0)
    x = torch.randn(T, H, device="cuda", generator=gen).bfloat16()
    logits = 1.5 * torch.randn(T, E, device="cuda", generator=gen)
    logits[:, 3] = -40.0  # an expert without rows
    w, idx = torch.topk(torch.softmax(logits, -1), k)
    run = (lambda: moe.routed(x, w, idx)) if v4 else (lambda: moe(x, logits))  # noqa: E731
    got = run()
    supported = I % 256 == 0  # (otherwise the down projection runs on the general kernel)
    name = bp.ext().last_kernel()
    assert ("+glu+gather" in name) == wide and (not wide or not supported or name == "gemm_tq2f4_i8+glu+gather+y16"), name
    tune("BP_TUNE_TQ2G", "b")
    ref = run()
    assert torch.isfinite(got).all()
    assert float((got.double() - ref.double()).norm() / ref.double().norm()) <= 4e-3  # (bf16 roundings and int8 steps that fall otherwise)


# 252 and 256 workgroups of 64 tokens x 256 rows, at a row length whose grouped calls keep to tiles of 32 there; the last tile of 1, 32 and 33 rows
@pytest.mark.parametrize("T,N,K,name", [(63 * 64 + 1, 1024, 3584, "gemm_tq2f4_i8"), (51 * 64 + 32, 1280, 3584, "gemm_tq2f4_i8"), (42 * 64 + 33, 1536, 1024, "gemm_tq2f4_i8"),
                                        (63 * 64, 1024, 3584, "gemm_tq2_i8_gs")])
def test_int8_linears_from_256_workgroups(T, N, K, name):
    import deepseekternarized_amd as bp

    gen = torch.Generator(device="cuda").manual_seed(22)
    (packed, scale), = _terms(1, N, K, 1, gen)
    x = torch.randn(T, K, device="cuda", generator=gen).bfloat16()
    lin = bp.TernaryLinear([bp.PackedTerm(packed[0], scale[0])], K, "tq2", 128)
    got = lin(x, torch.float32)
    assert bp.ext().last_kernel() == name, bp.ext().last_kernel()
    q, qs = bp.quant_act_int8(x)
    trits = bp.unpack(packed[0], "tq2", K).double()
    want = (q.double() @ (trits * scale[0].double().repeat_interleave(128, -1)).T) * qs.double().view(-1, 1)
    # exact sums of a group; K / 128 scaled additions in float32, each of which rounds by at most 2^-24 of a partial sum
    assert float((got.double() - want).norm() / want.norm()) <= K / 128 * 2.0**-24


@pytest.mark.parametrize("spread", [0, 12])
def test_bf16_pieces_keep_what_the_matrix_instruction_sums(tune, spread):
    """bf16 activations of one magnitude and over 2^12 of it: what a value loses below 2^-17 of its block's largest (the instruction
    aligns the products of 8 k to 13 bits below the largest; the first piece stays above that)."""
    import deepseekternarized_amd as bp

    T, N, K = 130, 1024, 2048
    gen = torch.Generator(device="cuda").manual_seed(23)
    (packed, scale), = _terms(1, N, K, 1, gen)
    x = torch.randn(T, K, device="cuda", generator=gen) * 2.0 ** -(spread * torch.rand(T, K, device="cuda", generator=gen))
    x = x.bfloat16()
    tune("BP_TUNE_TQ2G", "f")
    got = bp.TernaryLinear([bp.PackedTerm(packed[0], scale[0])], K, "tq2", 128, act="bf16")(x, torch.float32)
    assert bp.ext().last_kernel() == "gemm_tq2f4_bf16"
    want = x.double() @ (bp.unpack(packed[0], "tq2", K).double() * scale[0].double().repeat_interleave(128, -1)).T
    # an element's error is at most 2^-17.4 of its block's largest, uniform: 2^-19.2 of it in the mean square; that largest is
    # about 2.5 (spread 0: 0.3 % of the elements lose anything) to 4.5 (spread 12) times the root mean square
    bound = 2.5 * 2**-19.2 * 0.003**0.5 + 2**-22 if spread == 0 else 4.5 * 2**-19.2 + 2**-22
    assert float((got.double() - want).norm() / want.norm()) <= 2 * bound


# TQ1 layers either side of the lines from which their weights are rewritten as TQ2 ones: the same trits in either format are the same
# layer to the bit (int8: exact group sums; bf16: the same kernel, on which BP_TUNE_TQ2G=fp4 puts the TQ2 layer's down projection too). Rows that start at any byte; two terms; groups of 256.
@pytest.mark.parametrize("act,T,E,k,terms,group,H,I", [("int8", 383, 16, 2, 1, 128, 1280, 1024), ("int8", 384, 16, 2, 1, 128, 1280, 1024), ("int8", 300, 8, 3, 2, 128, 1024, 1792),
                                                       ("int8", 400, 8, 2, 1, 256, 2048, 2560), ("bf16", 3100, 8, 2, 2, 128, 1024, 1280)])
def test_tq1_layers_rewritten_as_tq2(tune, act, T, E, k, terms, group, H, I):
    import deepseekternarized_amd as bp
    from deepseekternarized_amd.moe import TernaryMoE

    gen = torch.Generator(device="cuda").manual_seed(24)

    def both(N, K):
        out = {"tq1": [], "tq2": []}
        for _ in range(terms):
            trits = torch.randint(-1, 2, (E * N, K), dtype=torch.int8, device="cuda", generator=gen)
            scale = (0.02 * torch.rand(E, N, K // group, device="cuda", generator=gen)).half()
            for fmt in out:
                out[fmt].append((bp.pack(trits, fmt).view(E, N, -1), scale))
        return out

    gate, up, down = both(I, H), both(I, H), both(H, I)
    x = torch.randn(T, H, device="cuda", generator=gen).bfloat16()
    logits = 1.5 * torch.randn(T, E, device="cuda", generator=gen)
    got = {}
    for fmt in gate:
        if act == "bf16" and fmt == "tq2":
            tune("BP_TUNE_TQ2G", "fp4")
        moe = TernaryMoE(gate[fmt], up[fmt], down[fmt], H, I, k, fmt, group, act=act)
        got[fmt] = moe(x, logits)
        rewritten = bp.ext().last_kernel().startswith("gemm_tq1_as_tq2f4")
        assert rewritten == (fmt == "tq1" and T * k >= (48 if act == "int8" and terms == 1 else 56 if act == "int8" else 84) * E), bp.ext().last_kernel()
        assert torch.equal(moe(x, logits), got[fmt])
    assert torch.isfinite(got["tq1"].float()).all() and torch.equal(got["tq1"], got["tq2"])


def test_tq1_layers_run_without_room_for_rewritten_weights(monkeypatch):
    """The rewriting's memory is optional: a device without it, and a capture (whose graph would keep it), run the layer on its TQ1
    weights - the same exact group sums, so the same bits."""
    import deepseekternarized_amd as bp
    from deepseekternarized_amd import moe as module

    gen = torch.Generator(device="cuda").manual_seed(28)
    H, I, E, k, T = 1024, 1024, 8, 2, 400

    def terms(N, K):
        trits = torch.randint(-1, 2, (E * N, K), dtype=torch.int8, device="cuda", generator=gen)
        return [(bp.pack(trits, "tq1").view(E, N, -1), (0.02 * torch.rand(E, N, K // 128, device="cuda", generator=gen)).half())]

    layer = module.TernaryMoE(terms(I, H), terms(I, H), terms(H, I), H, I, k, "tq1", 128, act="int8")
    x = torch.randn(T, H, device="cuda", generator=gen).bfloat16()
    logits = torch.randn(T, E, device="cuda", generator=gen)
    got = layer(x, logits)
    assert bp.ext().last_kernel().startswith("gemm_tq1_as_tq2f4_i8"), bp.ext().last_kernel()
    need = bp.ext().lib.bp_moe_layer_workspace_bytes(T, H, I, E, k, 0, 1)

    class Full:  # torch on a device with room for the layer's own workspace only
        def __getattr__(self, name):
            return getattr(torch, name)

        def empty(self, *size, **kw):
            if size[0] == need or kw.get("dtype") != torch.uint8:
                return torch.empty(*size, **kw)
            raise torch.cuda.OutOfMemoryError("no room")

    run = layer.graphed(T)
    assert torch.equal(run(x, logits), got) and torch.equal(run(x, logits), got)
    assert bp.ext().last_kernel().startswith("gemm_tq1f4_i8"), bp.ext().last_kernel()
    assert run.workspace.numel() == need
    monkeypatch.setattr(module, "torch", Full())
    assert torch.equal(layer(x, logits), got)
    assert bp.ext().last_kernel().startswith("gemm_tq1f4_i8"), bp.ext().last_kernel()


# TQ1 layers on that kernel as they are, by the byte table: tiles of 32 tokens, rows that start at any byte, windows of an odd count, two
# terms, groups of 256, scales of 32 bits (bf16 layers of these keep the kernel without pieces); either side of its lines. int8 (exact group sums): the bits of the same trits' TQ2 layer on the
# kernels over tiles of 32; bf16: of the kernel for 16 x 16 x 128 pieces, whose pieces and order of additions are the same.
@pytest.mark.parametrize("act,T,E,k,terms,group,H,I,sdt,name", [
    ("int8", 64, 64, 3, 1, 128, 1280, 1024, torch.float16, "gemm_tq1f4_i8"), ("int8", 65, 8, 2, 2, 128, 1792, 1280, torch.float16, "gemm_tq1f4_i8"),
    ("int8", 80, 4, 2, 1, 256, 2048, 2560, torch.float32, "gemm_tq1f4_i8"), ("int8", 64, 64, 2, 1, 128, 1280, 1024, torch.float16, None),
    ("bf16", 64, 8, 2, 1, 128, 1280, 1792, torch.bfloat16, "gemm_tq1f4_bf16"), ("bf16", 100, 4, 2, 1, 256, 2048, 2560, torch.float16, "gemm_tq1f4_bf16"),
    ("bf16", 180, 8, 2, 2, 128, 1024, 1280, torch.float16, "gemm_tq1f4_bf16"),
    ("bf16", 180, 8, 2, 2, 128, 1024, 1280, torch.float32, "gemm_tq1_bf16")])
def test_tq1_layers_by_the_byte_table(tune, act, T, E, k, terms, group, H, I, sdt, name):
    import deepseekternarized_amd as bp
    from deepseekternarized_amd.moe import TernaryMoE

    gen = torch.Generator(device="cuda").manual_seed(25)
    raw = [[(torch.randint(-1, 2, (E * N, K), dtype=torch.int8, device="cuda", generator=gen), (0.02 * torch.rand(E, N, K // group, device="cuda", generator=gen)).to(sdt))
            for _ in range(terms)] for N, K in ((I, H), (I, H), (H, I))]
    packed = lambda fmt: [[(bp.pack(t, fmt).view(E, s.shape[1], -1), s) for t, s in part] for part in raw]  # noqa: E731
    x = torch.randn(T, H, device="cuda", generator=gen).bfloat16()
    logits = 1.5 * torch.randn(T, E, device="cuda", generator=gen)
    logits[:, 1] = -40.0  # an expert without rows
    got = TernaryMoE(*packed("tq1"), H, I, k, "tq1", group, act=act)(x, logits)
    ran = bp.ext().last_kernel().split("+")[0]
    assert ran == name if name else "f4_" not in ran, ran
    if act == "int8":
        tune("BP_TUNE_F4", "1000000")
        ref = TernaryMoE(*packed("tq2"), H, I, k, "tq2", group, act=act)(x, logits)
    else:
        tune("BP_TUNE_F4Q", "1000000000")
        ref = TernaryMoE(*packed("tq1"), H, I, k, "tq1", group, act=act)(x, logits)
    assert torch.isfinite(got.float()).all() and torch.equal(got, ref), bp.ext().last_kernel()


# TQ2 layers with bf16 activations whose intermediate size is not half the hidden one: each product by its own line (768 tiles of 32 x 512), so
# that a layer between the two has one of them on the pieces and the other one on bf16 matrix instructions, over a tile list each. As
# grouped calls the products have the same lines, kernels and order of additions: the same bits.
@pytest.mark.parametrize("T,H,I,first,second", [(1015, 2048, 1536, False, False), (1030, 2048, 1536, True, False), (1530, 2048, 1536, True, True),
                                                (1015, 3072, 1024, False, False), (1030, 3072, 1024, False, True), (1530, 3072, 1024, True, True)])
@pytest.mark.parametrize("terms", [1, 2])
def test_bf16_layers_decide_per_product(tune, T, H, I, first, second, terms):
    from deepseekternarized_amd import ext
    from deepseekternarized_amd.moe import TernaryMoE

    gen = torch.Generator(device="cuda").manual_seed(27)
    E, k = 8, 4
    moe = TernaryMoE(_terms(E, I, H, terms, gen), _terms(E, I, H, terms, gen), _terms(E, H, I, terms, gen), H, I, k, "tq2", 128)
    x = torch.randn(T, H, device="cuda", generator=gen).bfloat16()
    logits = torch.randn(T, E, device="cuda", generator=gen)
    logits[:, 5] = -40.0  # an expert without rows
    got = moe(x, logits)
    name = ext().last_kernel()
    assert name.startswith("gemm_tq2f4_bf16" if second else "gemm_tq2_bf16") and ("+glu+gather" in name) == first, name
    assert torch.isfinite(got.float()).all() and torch.equal(got, moe.composed(x, logits)), name


# The tile list that the sort makes: one workgroup over more experts than it has threads, one over the whole list at 257 and 4095 rows, the
# two launches from 4096 on; experts without rows. Against the small-batch kernels, which take no list.
@pytest.mark.parametrize("T,E,k", [(300, 1030, 2), (129, 16, 2), (1365, 16, 3), (1366, 16, 3)])
def test_tile_lists_from_the_sort(tune, T, E, k):
    import deepseekternarized_amd as bp
    from deepseekternarized_amd.moe import TernaryMoE

    gen = torch.Generator(device="cuda").manual_seed(26)
    H = I = 1024  # noqa: E741
    moe = TernaryMoE(_terms(E, I, H, 1, gen), _terms(E, I, H, 1, gen), _terms(E, H, I, 1, gen), H, I, k, "tq2", 128)
    x = torch.randn(T, H, device="cuda", generator=gen).bfloat16()
    logits = 1.5 * torch.randn(T, E, device="cuda", generator=gen)
    logits[:, 5] = -40.0
    got = moe(x, logits)
    assert bp.ext().last_kernel().startswith("gemm_"), bp.ext().last_kernel()
    tune("BP_TUNE_TILES", "1000000")
    ref = moe(x, logits)
    assert torch.isfinite(got).all() and not bp.ext().last_kernel().startswith("gemm_tq2f4")
    assert float((got.double() - ref.double()).norm() / ref.double().norm()) <= 4e-3  # (sums in another order, each rounded to bf16 three times: 2^-9 once)
