"""The key parts vcpp_paged_prefill_split cuts a call into: the rule restated
(prefill_split_cost and its callers), by the chunks' real lengths where a chunk
can have several tiles (read back from a run's workspace in
test_prefill_split_gpu.py), by the host's bounds otherwise (read from what a
call says it needs where it is given no workspace).  And the sizes
vcpp_prefill_workspace_size gives for them."""
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


def tile_rows(dim):
    return 64 if dim <= 80 else 32


def most_parts(chunks, rows, prefix, heads, kv_heads, dim, cus=256):
    """prefill_most_splits."""
    tiles = -(-rows // tile_rows(dim)) * chunks * kv_heads * -(-(heads // kv_heads) // 4)
    return 1 if tiles >= 2 * cus else max(1, min(-(-2 * cus // tiles), (prefix + rows) // 512, 16))


def parts(lens, prefixes, heads, kv_heads, dim, cus=256, caps=None):
    """Parts of chunks of these lengths; caps: (max_chunk_len, max_prefix_len)."""
    rows, prefix = caps or (max(lens), max(prefixes))
    most = most_parts(len(lens), rows, prefix, heads, kv_heads, dim, cus)
    if most == 1 or len(lens) > 64:
        return most
    by_bounds = least_cost([rows] * len(lens), [prefix] * len(lens), heads, kv_heads, dim, cus, most)
    if not live(lens, by_bounds, most, rows, dim):
        return by_bounds
    keys = max(n + p for n, p in zip(lens, prefixes) if n > 0)
    return least_cost(lens, prefixes, heads, kv_heads, dim, cus, max(1, min(most, keys // 256)))


def live(lens, by_bounds, most, rows, dim):
    several = rows > tile_rows(dim)
    return several or by_bounds < most if len(lens) > 1 else several and by_bounds < most


def least_cost(lens, prefixes, heads, kv_heads, dim, cus, most):
    zh = kv_heads * -(-(heads // kv_heads) // 4)
    tiles = [-(-n // tile_rows(dim)) for n in lens]
    items = sum(tiles) * zh
    keys = max(n + p for n, p in zip(lens, prefixes) if n > 0)
    work = sum(t * (n + p) for t, n, p in zip(tiles, lens, prefixes)) * zh

    def cost(s):
        full, rest = divmod(items * s, 2 * cus)
        part = keys / (32 * s)
        return (min(part * (full + (0 if rest == 0 else 0.72 if rest <= cus else 1)), work / (64 * cus) + part / 2) +
                5 * (full + (rest > 0)) + (s * sum(lens) * heads * dim * 8 / 6.5e6 if s > 1 else 0))

    return min(range(1, most + 1), key=cost)


# (row counts, prefixes, heads, kv heads, head_dim)
@pytest.mark.parametrize("call,want", [
    (([50, 50, 50], [7000] * 3, 32, 8, 128), 10),     # 48 tiles: 11 parts would be 528 workgroups
    (([512], [32768], 64, 8, 80), 4),                 # 128 tiles: two per CU exactly
    (([300], [16384], 64, 8, 80), 6),                 # 80 tiles
    (([500] * 3, [8192] * 3, 64, 8, 80), 2),          # 384 tiles: a round and a half of halves beats one of wholes
    (([449, 387, 178], [18453, 19757, 14792], 24, 8, 80), 3),  # 144 real tiles of the grid's 192, which take two
    (([244, 357], [17221, 15921], 64, 8, 64), 3),
    (([2048] * 8, [1024] * 8, 64, 8, 80), 1),         # the chunks fill the GPU
    (([16], [400], 8, 8, 64), 1),                     # too short to cut
    (([16], [100000], 8, 1, 64), 16)])
def test_parts(call, want):
    assert parts(*call) == want


def test_one_chunk_loose_bounds():
    """A single chunk far shorter than its bound: the fullest count where that
    is the bound's best one, by the real lengths where it is not."""
    assert parts([100], [30000], 64, 8, 80, caps=(512, 32768)) == 4
    assert parts([100], [16000], 64, 8, 80, caps=(300, 16384)) == 7  # 6 by the bounds
    assert parts([90], [200], 64, 8, 80, caps=(300, 16384)) == 1


def test_workspace_asked():
    """A call asks for its own count's workspace where the host chose it, for
    the fullest count's where the device does."""
    for chunks in (1, 2, 5, 20, 65):
        for rows in (1, 31, 33, 64, 200):
            for prefix in (0, 700, 5000, 40000):
                for heads, kv_heads, dim in ((64, 8, 80), (28, 4, 128), (8, 8, 64), (1, 1, 64)):
                    most = most_parts(chunks, rows, prefix, heads, kv_heads, dim)
                    s = parts([rows] * chunks, [prefix] * chunks, heads, kv_heads, dim)
                    if most > 1 and chunks <= 64:
                        bounds = least_cost([rows] * chunks, [prefix] * chunks, heads, kv_heads, dim, 256, most)
                        s = most if live([rows] * chunks, bounds, most, rows, dim) else s
                    assert need(chunks, rows, prefix, heads, kv_heads, dim) == bytes_of(s, chunks, rows, heads, dim)


def test_size_at_caps_covers_smaller_calls():
    """A buffer sized once for an engine's limits, 512 rows of three chunks,
    holds shorter calls' partials; the size of every call is that of the
    fullest split, whose rows times parts do not jump with the rows."""
    cap = size(3, 512, 2000, 64, 8, 64)
    for rows in range(8, 513, 8):
        assert need(3, rows, 2000, 64, 8, 64) <= cap, rows
    for chunks in (1, 2, 3, 5):
        for rows in (1, 33, 64, 200, 320, 511, 512):
            for prefix in (0, 700, 2000, 5000, 40000):
                for heads, kv_heads, dim in ((64, 8, 80), (28, 4, 128), (8, 8, 64), (64, 8, 64)):
                    call = (chunks, rows, prefix, heads, kv_heads, dim)
                    assert size(*call) == bytes_of(most_parts(*call), chunks, rows, heads, dim), call
                    assert need(*call) <= size(*call), call
                    assert size(*call) <= 1024 * 256 * (4 * dim + 8) // (2 if dim == 128 else 1) + 256, call
