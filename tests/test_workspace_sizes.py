"""Workspace sizes that the library asks its callers for (no device needed)."""

import pytest

TQ1, TQ2 = 1, 2


@pytest.fixture(scope="module")
def lib():
    from deepseekternarized_amd.kernels import _lib

    if not _lib.LIB_PATH.exists():  # built only when nothing is there
        from deepseekternarized_amd.build import build

        build(verbose=False)
    return _lib.load()


# (lines of the kernel over tiles of 128 that k_gemm_f4 replaced) one expert: 96 tokens, 128 blocks, 192 with scales that leave room for one workgroup
# per CU (two terms from K = 1792, three always); several: 112 rows each and 384 blocks;
# scales that do not fit (K = 7168 in two terms), a group and row counts that the kernel does not take: no workspace
@pytest.mark.parametrize("T,N,K,group,E,fmt,terms,asks", [
    (2048, 2048, 2048, 128, 1, TQ2, 1, True), (1920, 2048, 2048, 128, 1, TQ2, 1, False), (2048, 2048, 2048, 128, 1, TQ2, 2, False), (3072, 2048, 2048, 128, 1, TQ2, 2, True),
    (2048, 2048, 1536, 128, 1, TQ2, 2, True), (2048, 2048, 1024, 128, 1, TQ2, 3, False), (8192, 2048, 4096, 128, 1, TQ2, 3, False), (8192, 2048, 7168, 128, 1, TQ2, 1, True),
    (8192, 2048, 7168, 128, 1, TQ2, 2, False), (8192, 2048, 2048, 64, 1, TQ2, 1, False), (8192, 2040, 2048, 128, 1, TQ2, 1, False), (8192, 2048, 2048, 256, 1, TQ2, 1, True),
    (20, 65536, 2048, 128, 1, TQ2, 1, False), (95, 65536, 2048, 128, 1, TQ2, 1, False), (96, 32768, 2048, 128, 1, TQ2, 1, True), (8192, 2048, 2048, 128, 1, TQ1, 1, False), (64 * 96, 2048, 2048, 128, 64, TQ2, 1, False), (64 * 112, 2048, 2048, 128, 64, TQ2, 1, True), (16 * 256, 2048, 2048, 128, 16, TQ2, 1, False)])
def test_int8_calls_ask_for_what_they_use(lib, T, N, K, group, E, fmt, terms, asks):
    assert (lib.bp_grouped_gemm_int8_workspace_bytes(T, N, K, group, E, fmt, terms, T) > 0) == asks


I8, BF16, F16, F32 = 0, 1, 2, 3


def _linear(lib, T, N, K, x=BF16, int8=0, out=BF16, fmt=TQ2, terms=1):
    return lib.bp_ternary_linear_workspace_bytes(x, int8, out, T, N, K, 128, fmt, terms)


def test_linears_ask_for_float32_rows_only_where_a_kernel_needs_them(lib):
    from deepseekternarized_amd.kernels import _lib

    assert (BF16, F16, F32, I8) == (_lib.BP_BF16, _lib.BP_F16, _lib.BP_F32, _lib.BP_I8)
    # bf16 rows from the kernel: as much as float32 rows from it
    for T, N, K, int8, fmt in [(8192, 6144, 2048, 1, TQ2), (8192, 6144, 2048, 0, TQ2), (200, 4096, 4096, 0, TQ2), (4096, 4096, 4096, 1, TQ1), (8192, 4096, 200, 0, TQ2)]:
        assert _linear(lib, T, N, K, int8=int8, fmt=fmt) == _linear(lib, T, N, K, int8=int8, fmt=fmt, out=F32)
    # TQ1 with few rows (a launch per term or segment), activations as a bf16 pair
    assert _linear(lib, 4, 2048, 7168, fmt=TQ1) == 4 * 4 * 2048
    assert _linear(lib, 512, 2048, 2048, x=F32) == _linear(lib, 512, 2048, 2048, x=F32, out=F32) + 4 * 512 * 2048


@pytest.mark.parametrize("int8,x,fmt", [(0, BF16, TQ2), (1, BF16, TQ2), (0, F32, TQ2), (0, BF16, TQ1), (1, F16, TQ1)])
def test_large_linears_ask_for_no_more_than_they_must(lib, int8, x, fmt):
    """Conversions of more than 8 GiB are left out, as in the grouped call: 4 Mi rows ask for their int8 rows at most."""
    T, K, N = 1 << 22, 7168, 8192
    assert _linear(lib, T, N, K, x=x, int8=int8, fmt=fmt) <= int8 * (T * K + 4 * T) + (N * K // 4 if fmt == TQ1 else 0) + 1024
    assert _linear(lib, T // 64, N, K, x=x, int8=int8, fmt=fmt) > int8 * (T * K + 4 * T) // 64 + (1 << 27)
    if x == F32:  # the bf16 pair still fits, its conversion does not
        assert _linear(lib, T // 16, N, K, x=x, int8=int8, fmt=fmt, out=F32) == 2 * 2 * T // 16 * K
    assert _linear(lib, 1 << 16, 1 << 21, 1 << 15, int8=1, fmt=TQ1, terms=2) < 6 << 30  # (17 GiB of weights a term)


def test_very_many_ids_sort_without_block_histograms(lib):
    """Beyond 8 Mi routed rows, where placing them block by block would read more than one workgroup sorting them takes: the
    layer's workspace loses the 8192 x 512 counters."""
    size = lambda T: lib.bp_moe_layer_workspace_bytes(T, 8, 8, 512, 8, BF16, TQ2)  # noqa: E731
    assert size((1 << 20) + 1) < size(1 << 20) - 4 * 8192 * 512 + (1 << 16)
