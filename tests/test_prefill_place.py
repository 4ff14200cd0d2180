"""The placement of prefill workgroups by the chunks' real lengths, restated
from live_work (vllm-cpp_amd/csrc/prefill.hip): every (tile, chunk, kv head and
head group) of the grid's tiles has exactly one workgroup, over ragged, empty
and over-long chunks and any prefix lengths, the live ones come first, and an
XCD whose share is at most one round of its CUs twice over puts no two heavy
tiles on one."""
import random

import pytest


def live_rank(tiles, lens, prefix, j, per, cus):
    if per <= cus or cus <= 0:
        return j
    if per <= 2 * cus:
        e = per - cus
        return cus - e + j if j < e else j - e if j < cus else per + cus - 1 - j
    if per <= 3 * cus and cus <= j < 2 * cus and sum(t * int((2 * p - n) / 32) for t, n, p in zip(tiles, lens, prefix)) < 0:
        return 3 * cus - 1 - j
    return j


def live_work(block, lens, prefix, max_chunk_len, rows, nz, cus):
    """(bx, by, bz) of workgroup `block`, or None."""
    nx = -(-max_chunk_len // rows)
    tiles = [max(0, min(-(-n // rows) if n > 0 else 0, nx)) for n in lens]
    block_x, q = block % nz, block // nz
    xcd, zz, nzx = block_x & 7, block_x >> 3, nz >> 3
    per, j = sum(tiles) * nzx, zz + nzx * q
    if j >= per:
        return None
    q, zz = divmod(live_rank(tiles, lens, prefix, j, per, cus), nzx)
    level = [max(int((p + n - 1) / rows), t - 1) for t, n, p in zip(tiles, lens, prefix)]
    l = max([v for v, t in zip(level, tiles) if t > 0] + [0])
    while True:
        live = [c for c, t in enumerate(tiles) if 0 <= level[c] - l < t]
        if q < len(live):
            break
        q -= len(live)
        l = l - 1 if live else max([v for v, t in zip(level, tiles) if t > 0 and v < l] + [0])
    return level[live[q]] - l, live[q], xcd * nzx + zz


def check(lens, prefix, max_chunk_len, rows, nz, cus):
    nx = -(-max_chunk_len // rows)
    blocks = nx * len(lens) * nz
    seen, share = {}, {}
    for b in range(blocks):
        w = live_work(b, lens, prefix, max_chunk_len, rows, nz, cus)
        if w is not None:
            assert w not in seen, (b, seen[w], w)
            seen[w] = b
        share.setdefault(b & 7, []).append(w)
    assert set(seen) == {(x, c, z) for c, n in enumerate(lens) for x in range(min(-(-max(n, 0) // rows), nx))
                         for z in range(nz)}
    for ws in share.values():
        live = [w is not None for w in ws]
        assert live == sorted(live, reverse=True)  # the live ones first
        ws = [w for w in ws if w is not None]
        if cus < len(ws) <= 2 * cus and min(prefix) >= 0:
            keys = [(prefix[c] + lens[c] - 1) // rows - x for x, c, _ in ws]
            pair = [keys[i] + keys[i + cus] for i in range(len(ws) - cus)]
            ranked = sorted(keys, reverse=True)
            light = ranked[2 * cus - len(ws):]
            best = [light[i] + light[-1 - i] for i in range(len(light) // 2)]
            assert sorted(pair) == sorted(best)


@pytest.mark.parametrize("seed", range(60))
def test_placement(seed):
    r = random.Random(seed)
    rows, nz = r.choice([32, 64]), 8 * r.randint(1, 3)
    chunks = r.choice([1, 2, 3, 4, 8, 13, 64])
    top = rows * r.randint(1, max(1, 48 * 32 // (nz * chunks))) - r.randint(0, rows - 1)
    lens = [r.choice([0, 1, top, r.randint(1, top), r.randint(1, top)]) for _ in range(chunks)]
    prefix = [r.choice([0, r.randint(0, 200), r.randint(0, 5000)]) for _ in lens]
    check(lens, prefix, top, rows, nz, 32)
    check([n + rows * 2 for n in lens], prefix, top, rows, nz, 32)          # longer than the caller said
    check(lens, [r.randint(-3000, 100) for _ in lens], top, rows, nz, 32)  # prefix lengths out of range
