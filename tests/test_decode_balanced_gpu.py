"""The balanced split (partition_size 0 on batches past the small-batch rule)
over the shapes of the page-staged kernel and of the register kernel: every
page type and head_dim, ragged and empty contexts, missing and out-of-pool
blocks, short tables, pages of 32 tokens, a reused workspace -- against the
oracle."""
import numpy as np
import pytest
import torch

import oracle_lib as O
import pyvcpp
from gpu_util import DevPool, assert_close, dev, gpu_decode
from test_decode_gpu import random_tables

pytestmark = pytest.mark.gpu

TOL = (2e-3, 1e-2)
KINDS = [O.ORC_F16, O.ORC_I8, O.ORC_FP8]
BASE = [0, 5, 16, 31, 300, 1025, 777, 64, 2000, 1, 511, 512, 513]


def contexts(H, Hkv, page):
    """Enough sequences that their partitions at the small-batch rule's longest
    (512 tokens, 1024 where the register kernel is the general path) are more
    than two workgroups per CU."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    pairs = Hkv * -(-(H // Hkv) // 8)
    parts = -(-max(BASE) // (512 if page else 1024))
    n = max(len(BASE), min(1000, 2 * cus) // (pairs * parts) + 1)
    assert n * pairs * parts > min(1000, 2 * cus)
    return np.array(BASE + [37 * i % 203 for i in range(n - len(BASE))], dtype=np.int32)


def check(kind, H, Hkv, D, page, seed):
    ctx = contexts(H, Hkv, page)
    nb = int(sum((int(c) + O.BS - 1) // O.BS for c in ctx)) + 6
    pool = O.make_pool(kind, seed, nb, Hkv, D)
    q = O.normal(seed + 1, (len(ctx), H, D))
    tables = random_tables(seed + 2, ctx, nb)
    lens = np.full(len(ctx), tables.shape[1], dtype=np.int32)
    dp = DevPool(pool)
    for skips in (False, True) if kind == O.ORC_F16 else (True,):
        if skips:
            tables[4, 3], tables[5, 40], tables[8, 0], tables[8, 124] = -1, nb + 100, -5, 10 ** 6
            lens[6], lens[7], lens[11] = 20, 0, 31
        want = O.decode(pool, q, tables, ctx, H, table_lens=lens)
        got = gpu_decode(dp, q, tables, ctx, H, table_lens=lens)
        assert_close(got, want, *TOL, what="balanced kind=%d H=%d/%d D=%d skips=%d" % (kind, H, Hkv, D, skips))
        assert np.all(got[ctx == 0] == 0.0)


@pytest.mark.parametrize("heads,D", [((16, 16), 80)] + [(h, D) for h in ((64, 8), (32, 4), (16, 4), (24, 8))
                                                        for D in (64, 80, 128)])
@pytest.mark.parametrize("kind", KINDS)
def test_page_kernel(cuda, kind, heads, D):
    check(kind, heads[0], heads[1], D, True, 6000 + D + heads[0])


@pytest.mark.parametrize("heads,D", [((12, 2), 64), ((12, 2), 80), ((12, 2), 128), ((40, 2), 80), ((7, 1), 128),
                                     ((18, 6), 64)])
@pytest.mark.parametrize("kind", KINDS)
def test_register_kernel(cuda, kind, heads, D):
    check(kind, heads[0], heads[1], D, False, 6200 + D + heads[0])


@pytest.mark.parametrize("heads", [(64, 8), (12, 2)])
def test_block_size_32(cuda, heads):
    """Pages of 32 tokens: a 16-token tile is half a page."""
    (H, Hkv), bs, D = heads, 32, 80
    ctx = contexts(H, Hkv, Hkv % 4 == 0)
    nbs = [(int(c) + bs - 1) // bs for c in ctx]
    nb = sum(nbs) + 5
    k, v = (O.f16_trunc(O.normal(6400 + i, (nb, bs, Hkv, D))) for i in range(2))
    perm = O.permutation(6402, nb)
    tables = np.full((len(ctx), max(nbs)), -1, np.int32)
    at = 0
    for i, n in enumerate(nbs):
        tables[i, :n] = perm[at:at + n]
        at += n
    q = O.normal(6403, (len(ctx), H, D))
    pool = O.Pool(O.ORC_F16, k, v, block_size=bs)
    want = O.decode(pool, q, tables, ctx, H)
    got = gpu_decode(DevPool(pool), q, tables, ctx, H)
    assert_close(got, want, *TOL, what="balanced block size 32 H=%d/%d" % heads)


@pytest.mark.parametrize("heads", [(64, 8), (12, 2)])
def test_workspace_reuse(cuda, heads):
    """One workspace across calls with changing q and lengths: no call may see
    another's partials."""
    H, Hkv = heads
    ctx = contexts(H, Hkv, Hkv % 4 == 0)
    nb = 2 * int(sum((int(c) + O.BS - 1) // O.BS for c in ctx)) + 8
    pool = O.make_pool(O.ORC_F16, 6500, nb, Hkv, 80)
    dp = DevPool(pool)
    need = pyvcpp.decode_workspace_size(dp.pages, len(ctx), H, int(ctx.max()))
    ws = torch.zeros(max(need, 1), dtype=torch.uint8, device="cuda:0")
    for it in range(4):
        ctx = np.roll(ctx, 5)
        tables = random_tables(6510 + it, ctx, nb)
        q = O.normal(6520 + it, (len(ctx), H, 80))
        out = torch.full((len(ctx), H, 80), float("nan"), device="cuda:0")
        pyvcpp.paged_decode(dp.pages, dev(q), out, dev(tables), dev(ctx), int(ctx.max()), H, workspace=ws)
        torch.cuda.synchronize()
        assert_close(out.cpu().numpy(), O.decode(pool, q, tables, ctx, H), *TOL, what="balanced reuse it=%d" % it)
