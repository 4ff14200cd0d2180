"""The key parts vcpp_paged_prefill_split cuts a call into, read from what it
says it needs where it is given no workspace: never more than fill two
workgroups per CU, none that spills a few workgroups into a round of their
own.  And the sizes vcpp_prefill_workspace_size gives for them."""
import ctypes
import re

import pytest
import torch

import pyvcpp


def _pages(kv_heads, dim):
    base = 4096  # never read: no call here reaches a GPU
    return pyvcpp.KVPages(pyvcpp.KV_F16, 16, kv_heads, dim, 0, 16 * kv_heads * dim, 0, base, base, None, None)


def bytes_of(s, chunks, rows, heads, dim):
    n = chunks * rows * heads
    return 0 if s == 1 else (s * n * dim * 4 + 255) // 256 * 256 + s * n * 8


def size(chunks, rows, prefix, heads, kv_heads, dim):
    return pyvcpp.prefill_workspace_size(_pages(kv_heads, dim), chunks, rows, prefix, heads)


def need(chunks, rows, prefix, heads, kv_heads, dim):
    """Bytes the call itself asks for (0: it goes on to its launch, an error
    without a GPU)."""
    if torch.cuda.device_count() > 0:
        pytest.skip("an unsplit call would launch")
    p = 4096
    rc = pyvcpp.lib().vcpp_paged_prefill_split(ctypes.byref(_pages(kv_heads, dim)), p, p, p, 64, p, p, chunks, rows,
                                               prefix, heads, None, 0, None)
    if rc != pyvcpp.VCPP_E_WORKSPACE:
        assert rc == pyvcpp.VCPP_E_HIP, pyvcpp.last_error()
        return 0
    return int(re.search(r"needs (\d+) workspace bytes", pyvcpp.last_error()).group(1))


def parts(chunks, rows, prefix, heads, kv_heads, dim):
    got = need(chunks, rows, prefix, heads, kv_heads, dim)
    for s in range(1, 17):
        if got == bytes_of(s, chunks, rows, heads, dim):
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


def test_size_at_caps_covers_smaller_calls():
    """A buffer sized once for an engine's limits: 512 rows and 320 rows of
    three chunks (one part and two), and the size of every call is that of
    the fullest split, whose rows times parts do not jump with the rows."""
    cap = size(3, 512, 2000, 64, 8, 64)
    for rows in range(8, 513, 8):
        assert need(3, rows, 2000, 64, 8, 64) <= cap, rows
    for chunks in (1, 2, 3, 5):
        for rows in (1, 33, 64, 200, 320, 511, 512):
            for prefix in (0, 700, 2000, 5000, 40000):
                for heads, kv_heads, dim in ((64, 8, 80), (28, 4, 128), (8, 8, 64), (64, 8, 64)):
                    tiles = -(-rows // (64 if dim <= 80 else 32)) * chunks * kv_heads * -(-(heads // kv_heads) // 4)
                    most = 1 if tiles >= 512 else max(1, min(-(-512 // tiles), (prefix + rows) // 512, 16))
                    call = (chunks, rows, prefix, heads, kv_heads, dim)
                    assert size(*call) == bytes_of(most, chunks, rows, heads, dim), call
                    assert need(*call) <= size(*call), call
                    assert size(*call) <= 1024 * 256 * (4 * dim + 8) // (2 if dim == 128 else 1) + 256, call
