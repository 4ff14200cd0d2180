"""The split-K merge kernels at the edges of their rule: 8, 2 and 1 waves per
256 outputs, one fragment to hundreds, fragment counts around the chunk of 8,
odd query groups and head dims that leave a partial unit, and an output that
is only 4-byte aligned -- against the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle_lib as O
import pyvcpp
from gpu_util import DevPool, assert_close, dev

pytestmark = pytest.mark.gpu

TOL = {O.ORC_F32: (1e-4, 1e-4), O.ORC_F16: (2e-3, 1e-2), O.ORC_FP8: (2e-3, 1e-2)}


def _run(kind, ctx, H, Hkv, D, partition, seed):
    ctx = np.asarray(ctx, dtype=np.int32)
    used = [(int(c) + O.BS - 1) // O.BS for c in ctx]
    nb = sum(used) + 3
    pool = O.make_pool(kind, seed, nb, Hkv, D)
    q = O.normal(seed + 1, (len(ctx), H, D))
    perm = O.permutation(seed + 2, nb)
    tables = np.full((len(ctx), max(used)), -1, dtype=np.int32)
    at = 0
    for i, n in enumerate(used):
        tables[i, :n] = perm[at:at + n]
        at += n
    want = O.decode(pool, q, tables, ctx, H)
    dp = DevPool(pool)
    qd = dev(q)
    flat = torch.full((qd.numel() + 1,), float("nan"), device=qd.device)
    out = flat[1:].view(qd.shape)  # 4-byte aligned only
    pyvcpp.paged_decode(dp.pages, qd, out, dev(tables), dev(ctx), int(ctx.max()), H, partition_size=partition)
    torch.cuda.synchronize()
    assert torch.isnan(flat[0])
    assert_close(out.cpu().numpy(), want, *TOL[kind], what="merge kind=%d n=%d H=%d/%d D=%d P=%d"
                 % (kind, len(ctx), H, Hkv, D, partition))


ONE = [5003]
SOME = [1 + (37 * i * i + 11) % 611 for i in range(40)]
MANY = [1 + (53 * i * i + 7) % 301 for i in range(96)]


@pytest.mark.parametrize("partition", [0, 16])
@pytest.mark.parametrize("ctx,H,Hkv,D", [
    (ONE, 64, 8, 80), (ONE, 28, 4, 128), (ONE, 3, 1, 64), ([64], 64, 8, 80), ([130], 24, 8, 64),
    (SOME, 64, 8, 80), (SOME, 12, 2, 128), (MANY, 64, 8, 80), (MANY, 32, 8, 128)])
def test_split_merge(cuda, ctx, H, Hkv, D, partition):
    _run(O.ORC_F16, ctx, H, Hkv, D, partition, 4100 + D + H)


@pytest.mark.parametrize("partition", [0, 64])
@pytest.mark.parametrize("n,long,H,Hkv,D", [
    (129, 3001, 64, 8, 80), (200, 700, 28, 4, 128), (450, 90, 12, 2, 128), (300, 5003, 8, 8, 64), (600, 2100, 20, 2, 64)])
def test_split_merge_many(cuda, n, long, H, Hkv, D, partition):
    """Many sequences, a workgroup per (sequence, kv-head slot): more lengths
    than its waves scan in a round, empty ones among them, one sequence over
    many ranges, slots of fewer units than waves."""
    ctx = [(29 * i * i + 5) % 67 for i in range(n)]
    ctx[n // 3] = long
    _run(O.ORC_F16, ctx, H, Hkv, D, partition, 4200 + n)


def test_split_merge_fp8(cuda):
    _run(O.ORC_FP8, SOME, 64, 8, 80, 0, 4300)


@pytest.mark.parametrize("partition", [0, 16, 256])
@pytest.mark.parametrize("ctx,H,Hkv,D", [
    (ONE, 8, 2, 80), ([257], 3, 3, 20), (SOME, 12, 2, 100), (MANY, 64, 8, 64)])
def test_parts_merge(cuda, ctx, H, Hkv, D, partition):
    _run(O.ORC_F32, ctx, H, Hkv, D, partition, 4500 + D + H)
