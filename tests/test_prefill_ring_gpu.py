"""fp16 prefill around the K/V ring's lengths: key counts of one block to a
few past the ring's depth, odd and even, whole and ragged, at each ring shape
(6 stages taken two per barrier, 4 stages taken one), against the oracle."""
import pytest

import oracle_lib as O
from gpu_util import DevPool, assert_close, gpu_prefill
from test_prefill_gpu import ATOL, RTOL, make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 80, 128])
def test_ring_lengths(cuda, D):
    keys = [1, 32, 33, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 225, 257]
    chunk = [min(n, 1 + 7 * i % 40) for i, n in enumerate(keys)]
    prefix = [n - m for n, m in zip(keys, chunk)]
    pool, q16, q32, tables, q_start, pre = make_case(O.ORC_F16, 930 + D, prefix, chunk, 8, 2, D)
    want = O.prefill(pool, q32, tables, q_start, pre, 8)
    got = gpu_prefill(DevPool(pool), q16, tables, q_start, pre, 8)
    assert_close(got, want, ATOL, RTOL, what="prefill ring D=%d" % D)


def test_ring_pairs(cuda):
    """head_dim 128, few enough workgroups over long enough tables that the
    4-stage ring takes two blocks per barrier: odd and even block counts, short
    chunks beside long ones; one chunk, and several of more than one tile."""
    keys = [1, 33, 64, 65, 129, 1023, 1024, 1025, 1056, 1057, 1089, 1120]
    chunk = [min(n, 1 + 7 * i % 40) for i, n in enumerate(keys)]
    for lo, hi in ((0, 12), (11, 12)):
        prefix = [n - m for n, m in zip(keys[lo:hi], chunk[lo:hi])]
        for H, Hkv in ((8, 2), (8, 8)):
            pool, q16, q32, tables, q_start, pre = make_case(O.ORC_F16, 950 + hi, prefix, chunk[lo:hi], H, Hkv, 128)
            want = O.prefill(pool, q32, tables, q_start, pre, H)
            got = gpu_prefill(DevPool(pool), q16, tables, q_start, pre, H)
            assert_close(got, want, ATOL, RTOL, what="prefill ring pairs %d..%d H=%d/%d" % (lo, hi, H, Hkv))
