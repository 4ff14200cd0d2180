"""Prefill grids around the edges of the workgroup order's rule (one round of
the CUs, two, six, past it; chunk counts that divide a round and not), chunks
of very uneven length: a workgroup placed twice or not at all leaves rows
unwritten.  Against the oracle."""
import pytest

import oracle_lib as O
from gpu_util import DevPool, assert_close, gpu_prefill
from test_prefill_gpu import ATOL, RTOL, make_case

pytestmark = pytest.mark.gpu


# tiles of 32 tokens; 8 kv heads: tiles x chunks workgroups per XCD
@pytest.mark.parametrize("tiles,chunks,heads", [
    (1, 1, 8), (4, 8, 8), (11, 3, 8), (8, 8, 8), (5, 13, 8), (24, 8, 8), (25, 8, 8), (7, 6, 64), (6, 4, 64)])
def test_order(cuda, tiles, chunks, heads):
    chunk = [max(1, 32 * tiles - 3 if i == chunks // 2 else (i * 37) % (20 * tiles)) for i in range(chunks)]
    prefix = [(i * 29) % 50 for i in range(chunks)]
    pool, q16, q32, tables, q_start, pre = make_case(O.ORC_F16, 960 + tiles, prefix, chunk, heads, 8, 128)
    want = O.prefill(pool, q32, tables, q_start, pre, heads)
    got = gpu_prefill(DevPool(pool), q16, tables, q_start, pre, heads)
    assert_close(got, want, ATOL, RTOL, what="prefill order %d x %d, %d heads" % (tiles, chunks, heads))
