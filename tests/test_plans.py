"""Launch plans seen from the host (CPU): what the workspace queries ask for.
Without a device the plans are made for 256 CUs."""
import threading

import pytest

from mtp_hip import _lib as L


@pytest.fixture(scope="module")
def lib():
    return L.load()


@pytest.mark.parametrize("dtype,D", [(L.F32, 64), (L.F32, 128), (L.BF16, 256)])
@pytest.mark.parametrize("keys", [64 * 64, 64 * 64 + 1, 64 * 65537, 2 ** 31 - 2 ** 21])
@pytest.mark.parametrize("chunk", [1, 3, 10 ** 6])
def test_decode_attention_has_at_most_64_chunks(lib, dtype, D, keys, chunk):
    """Also with the chunk length set: counters, then (O, max, sum) of a chunk
    for each of three heads."""
    with L.tuning(attn_chunk_blocks=chunk):
        n = lib.mtp_attention_workspace_bytes(dtype, 1, 1, 3, D, 0, keys)
    most = L.MTP_COUNTER_BYTES + 3 * 64 * (D + 2) * 4
    assert n <= -(-most // 256) * 256


def test_kept_decode_plans_are_of_their_sizes_and_keys(lib):
    """The plans a thread keeps: more sizes than it holds, asked for in both
    orders, against a thread that has none; a tuning key set in between. At more
    than 128 heads the MFMA kernel's plan has one chunk and no workspace, so the
    query shows the decode kernel's chunks."""
    sizes = [(H, D, keys) for D in (64, 128) for H in (160, 257, 288, 384)
             for keys in (65, 511, 700, 1024, 1500, 2272, 4096)]

    def ask(size):
        H, D, keys = size
        return lib.mtp_attention_workspace_bytes(L.BF16, 1, 1, H, D, 0, keys)

    def ask_anew(size):
        got = []
        t = threading.Thread(target=lambda: got.append(ask(size)))
        t.start()
        t.join()
        return got[0]

    fresh = {size: ask_anew(size) for size in sizes}
    assert len(set(fresh.values())) > 8  # plans of several chunk counts
    assert [ask(s) for s in sizes] == [fresh[s] for s in sizes]
    assert [ask(s) for s in sizes[::-1]] == [fresh[s] for s in sizes[::-1]]
    last = sizes[-1]
    with L.tuning(attn_chunk_blocks=1):
        assert ask(last) == ask_anew(last) != fresh[last]
    assert ask(last) == fresh[last]


@pytest.mark.parametrize("w", [L.BF16, L.FP8E4M3])
@pytest.mark.parametrize("M,K", [(16384, 4096), (16385, 4096), (32768, 8192), (10 ** 6, 4096),
                                 (65, 262144), (1000, 262208)])
@pytest.mark.parametrize("N", [64, 14336])
def test_long_prompts_keep_a_bounded_workspace(lib, M, N, K, w):
    """x * gamma of at most 128 MiB at a time, beside the counters, the row
    factors and the sums of K-splits (two 128 x 128 fp32 tiles per CU)."""
    most = L.MTP_COUNTER_BYTES + (128 << 20) + 4 * M + 256 * 2 * 128 * 128 * 4 + 1024
    assert lib.mtp_rmsnorm_linear_workspace_bytes(L.BF16, w, M, N, K) <= most


@pytest.mark.parametrize("w", [L.BF16, L.FP8E4M3])
@pytest.mark.parametrize("M,N,K,narrow", [(4096, 64, 4096, True), (1000, 100, 3200, True),
                                          (999, 64, 4096, False), (4096, 64, 768, False),
                                          (4096, 512, 4096, False)])
def test_many_rows_of_few_columns_stay_on_the_row_chunk_kernel(lib, w, M, N, K, narrow):
    """Their workspace has no room for x * gamma of every row."""
    both = lib.mtp_rmsnorm_linear_workspace_bytes(L.BF16, w, M, N, K)
    assert (both < M * K * 2) == narrow
    with L.tuning(pg=0):
        assert both >= lib.mtp_rmsnorm_linear_workspace_bytes(L.BF16, w, M, N, K)
