"""The small-batch decode kernel (partition_size 0 on small batches) over the
forms it accepts: contexts around its tile, its waves and its partitions,
empty ones, short and missing table entries, every page type and head shape,
page sizes, and lengths past the host's bound -- against the oracle, and
against the fixed-partition path on the same inputs."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_util import DevPool, assert_close, gpu_decode

pytestmark = pytest.mark.gpu

TOL = (2e-3, 1e-2)


def _tables(seed, ctx, nb, bs):
    used = [(int(c) + bs - 1) // bs for c in ctx]
    perm = O.permutation(seed, nb)
    t = np.full((len(ctx), max(max(used), 1)), -1, dtype=np.int32)
    at = 0
    for i, n in enumerate(used):
        t[i, :n] = perm[at:at + n]
        at += n
    return t, at


def _check(kind, ctx, H, Hkv, D, seed, table_lens=None, spoil=None, max_context_len=None):
    ctx = np.asarray(ctx, dtype=np.int32)
    nb = sum((int(c) + O.BS - 1) // O.BS for c in ctx) + 4
    pool = O.make_pool(kind, seed, nb, Hkv, D)
    q = O.normal(seed + 1, (len(ctx), H, D))
    tables, _ = _tables(seed + 2, ctx, nb, O.BS)
    for (i, j, v) in spoil or ():
        tables[i, j] = v
    seen = ctx if max_context_len is None else np.minimum(ctx, max_context_len).astype(np.int32)
    want = O.decode(pool, q, tables, seen, H, table_lens=table_lens)
    dp = DevPool(pool)
    what = "small kind=%d n=%d H=%d/%d D=%d" % (kind, len(ctx), H, Hkv, D)
    got = gpu_decode(dp, q, tables, ctx, H, table_lens=table_lens, max_context_len=max_context_len)
    assert_close(got, want, *TOL, what=what)
    fixed = gpu_decode(dp, q, tables, ctx, H, table_lens=table_lens, partition_size=64, max_context_len=max_context_len)
    assert_close(got, fixed, 2e-5, 2e-5, what=what + " vs P=64")
    assert np.all(got[seen == 0] == 0.0)


KINDS = [O.ORC_F16, O.ORC_I8, O.ORC_FP8]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("D", [64, 80, 128])
def test_context_edges(cuda, kind, D):
    """One partition: lengths around a tile, a wave round and 256."""
    _check(kind, [0, 1, 15, 16, 17, 63, 64, 65, 127, 130, 255, 256], 16, 2, D, 5000 + D)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("ctx", [[257], [64 * 9, 1, 0, 64 * 9 - 1], [1500, 3, 700, 2047], [4100, 5, 900]])
def test_partitions(cuda, kind, ctx):
    """Several partitions, some sequences ending before them, one of no token."""
    _check(kind, ctx, 32, 8, 128, 5100)
    _check(kind, ctx, 64, 8, 80, 5200)


@pytest.mark.parametrize("H,Hkv", [(8, 8), (24, 8), (7, 1), (12, 2), (18, 6), (40, 2), (33, 3)])
def test_head_shapes(cuda, H, Hkv):
    """Odd groups, groups over 8 heads, kv heads the page-staged kernel does
    not take (whose partitions go up to 1024 tokens)."""
    _check(O.ORC_F16, [300, 17, 1000], H, Hkv, 80, 5300 + H)
    _check(O.ORC_I8, [90] * 30 + [2600] * 3, H, Hkv, 64, 5400 + H)


@pytest.mark.parametrize("n", [1, 7, 8, 9, 17])
@pytest.mark.parametrize("H,Hkv", [(6, 1), (12, 3), (64, 8)])
def test_workgroup_order(cuda, n, H, Hkv):
    """(sequence, partition) counts around the rounds of eight XCDs."""
    _check(O.ORC_F16, [200 + i for i in range(n)], H, Hkv, 80, 5450 + n)      # one partition
    _check(O.ORC_F16, [700 - 90 * (i % 5) for i in range(n)], H, Hkv, 80, 5470 + n)


def test_one_long_sequence(cuda):
    """Over 128 partitions of 64 and 128 tokens: the rule takes longer ones."""
    _check(O.ORC_F16, [33001], 12, 2, 128, 5490)


@pytest.mark.parametrize("kind", KINDS)
def test_skips(cuda, kind):
    """Short tables, missing and out-of-pool blocks, a length past the bound."""
    ctx = [400, 130, 700, 40]
    _check(kind, ctx, 16, 2, 80, 5500, table_lens=np.array([25, 3, 44, 0], dtype=np.int32),
           spoil=[(0, 1, -1), (0, 24, 10 ** 6), (2, 0, -1), (2, 43, -5)])
    _check(kind, ctx, 16, 2, 80, 5600, max_context_len=333)


def test_block_sizes(cuda):
    """Pages of 32 and 48 tokens hold the same rows as pages of 16."""
    import torch
    import pyvcpp
    H, Hkv, D, ctx = 16, 2, 80, [500, 33, 96, 1]
    rows = max(ctx)
    k = O.normal(5700, (len(ctx), rows, Hkv, D)).astype(np.float16)
    v = O.normal(5701, (len(ctx), rows, Hkv, D)).astype(np.float16)
    q = torch.from_numpy(O.normal(5702, (len(ctx), H, D))).cuda()
    outs = []
    for bs in (16, 32, 48):
        per = -(-rows // bs)
        pad = lambda x: np.concatenate([x, np.zeros((len(ctx), per * bs - rows, Hkv, D), np.float16)], 1)
        kp, vp = (torch.from_numpy(pad(x).reshape(-1, bs, Hkv, D)).cuda() for x in (k, v))
        tables = torch.arange(len(ctx) * per, dtype=torch.int32, device="cuda").view(len(ctx), per)
        pages = pyvcpp.kv_pages(pyvcpp.KV_F16, kp, vp, bs, Hkv, D, len(ctx) * per, bs * Hkv * D)
        out = torch.empty_like(q)
        pyvcpp.paged_decode(pages, q, out, tables, torch.tensor(ctx, dtype=torch.int32, device="cuda"), max(ctx), H)
        outs.append(out.cpu().numpy())
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])
    assert np.isfinite(outs[0]).all()


def test_int8_small_scales(cuda):
    """V scales near 2^-11: P times a scale keeps its 22 bits (about 2e-7
    here with fp32 sums of 300 terms; low parts lost to fp16's subnormals
    would show 3e-5)."""
    ctx = np.array([300, 41, 256], dtype=np.int32)
    pool = O.make_pool(O.ORC_I8, 5800, 64, 8, 80, 0.0, 0.02)
    q = O.normal(5801, (3, 64, 80))
    tables, _ = _tables(5802, ctx, 64, O.BS)
    want = O.decode(pool, q, tables, ctx, 64)
    got = gpu_decode(DevPool(pool), q, tables, ctx, 64)
    assert np.linalg.norm(got - want) <= 3e-6 * np.linalg.norm(want)
