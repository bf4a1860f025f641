"""Launch plans seen from the host (CPU): what the workspace queries ask for.
Without a device the plans are made for 256 CUs."""
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
