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


# one expert: 128 blocks as four waves, 192 as eight (two terms from K = 1792, three always); several: 112 rows each and 384 blocks;
# scales that do not fit (K = 7168 in two terms), a group and row counts that the kernel does not take: no workspace
@pytest.mark.parametrize("T,N,K,group,E,fmt,terms,asks", [
    (2048, 2048, 2048, 128, 1, TQ2, 1, True), (1920, 2048, 2048, 128, 1, TQ2, 1, False), (2048, 2048, 2048, 128, 1, TQ2, 2, False), (3072, 2048, 2048, 128, 1, TQ2, 2, True),
    (2048, 2048, 1536, 128, 1, TQ2, 2, True), (2048, 2048, 1024, 128, 1, TQ2, 3, False), (8192, 2048, 4096, 128, 1, TQ2, 3, False), (8192, 2048, 7168, 128, 1, TQ2, 1, True),
    (8192, 2048, 7168, 128, 1, TQ2, 2, False), (8192, 2048, 2048, 64, 1, TQ2, 1, False), (8192, 2040, 2048, 128, 1, TQ2, 1, False), (8192, 2048, 2048, 256, 1, TQ2, 1, True),
    (8192, 2048, 2048, 128, 1, TQ1, 1, False), (64 * 96, 2048, 2048, 128, 64, TQ2, 1, False), (64 * 112, 2048, 2048, 128, 64, TQ2, 1, True), (16 * 256, 2048, 2048, 128, 16, TQ2, 1, False)])
def test_int8_calls_ask_for_what_they_use(lib, T, N, K, group, E, fmt, terms, asks):
    assert (lib.bp_grouped_gemm_int8_workspace_bytes(T, N, K, group, E, fmt, terms, T) > 0) == asks
