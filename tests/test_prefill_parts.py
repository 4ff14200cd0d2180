"""The key parts vcpp_paged_prefill_split cuts a call into, read back from its
workspace size: never more than fill two workgroups per CU, none that spills
a few workgroups into a round of their own."""
import pytest

import pyvcpp


def parts(chunks, rows, prefix, heads, kv_heads, dim):
    pages = pyvcpp.KVPages(pyvcpp.KV_F16, 16, kv_heads, dim, 0, 16 * kv_heads * dim, 0, None, None, None, None)
    got = pyvcpp.prefill_workspace_size(pages, chunks, rows, prefix, heads)
    if got == 0:
        return 1
    n = chunks * rows * heads
    for s in range(2, 17):
        if got == (s * n * dim * 4 + 255) // 256 * 256 + s * n * 8:
            return s
    raise AssertionError("workspace of %d bytes is no whole number of parts" % got)


# (chunks, rows, prefix, heads, kv heads, head_dim) on 256 CUs (what the
# library assumes where there is no GPU to ask)
@pytest.mark.parametrize("call,want", [
    ((3, 50, 7000, 32, 8, 128), 10),     # 48 tiles: 11 parts would be 528 workgroups
    ((1, 512, 32768, 64, 8, 80), 4),     # 128 tiles: two per CU exactly
    ((1, 300, 16384, 64, 8, 80), 6),     # 80 tiles
    ((3, 500, 8192, 64, 8, 80), 2),      # 384 tiles: a round and a half of halves beats one of wholes
    ((8, 2048, 1024, 64, 8, 80), 1),     # the chunks fill the GPU
    ((1, 16, 400, 8, 8, 64), 1),         # too short to cut
    ((1, 16, 100000, 8, 1, 64), 16)])
def test_parts(call, want):
    assert parts(*call) == want


def test_parts_bound():
    """Never more parts than fill two workgroups per CU, so the workspace is
    within what that count needs; whole tiles only."""
    for chunks in (1, 2, 5):
        for rows in (1, 33, 64, 200, 511):
            for prefix in (0, 700, 5000, 40000):
                for heads, kv_heads, dim in ((64, 8, 80), (28, 4, 128), (8, 8, 64)):
                    tiles = -(-rows // (64 if dim <= 80 else 32)) * chunks * kv_heads * -(-(heads // kv_heads) // 4)
                    most = max(1, min(-(-512 // tiles), (prefix + rows) // 512, 16))
                    assert 1 <= parts(chunks, rows, prefix, heads, kv_heads, dim) <= most
