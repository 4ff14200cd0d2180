"""flash_attention_cuda with a pair's keys split over workgroups: key counts
around the parts' 64-key rounds and the rule's edges, a part longer than the
4096-key logit segment, masks (whole parts masked too), every head_dim of the
one-pass kernel -- against the oracle."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_util import assert_close
from test_dense_gpu import run_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("shape", [
    (1, 1, 1, 1024, 64), (1, 3, 2, 2047, 64), (2, 4, 1, 2049, 80), (1, 8, 1, 1025, 128), (1, 2, 1, 4200, 96),
    (1, 1, 3, 70001, 64),        # 16 parts of over 4096 keys
    (4, 32, 1, 4100, 64),        # two parts a pair
    (1, 300, 1, 4096, 64)])      # a short second round of workgroups
def test_split(cuda, shape, masked):
    B, H, ql, kv, D = shape
    q, k, v = O.normal(81, (B, H, ql, D)), O.normal(82, (B, H, kv, D)), O.normal(83, (B, H, kv, D))
    mask = None
    if masked:
        mask = np.where(O.normal(84, (kv,)) > 0.0, 0.0, -1.0).astype(np.float32)
        mask[: kv // 3] = -1.0
    want, want_w = O.flash(q, k, v, mask)
    got, got_w = run_gpu(q, k, v, mask)
    assert_close(got, want, 1e-4, 1e-4, what="flash split out %s" % (shape,))
    assert_close(got_w, want_w, 1e-5, 1e-4, what="flash split weights %s" % (shape,))
    if masked:
        assert np.all(got_w[:, mask < 0] == 0.0)


def test_split_all_masked(cuda):
    q, k, v = O.normal(91, (1, 2, 1, 80)), O.normal(92, (1, 2, 1500, 80)), O.normal(93, (1, 2, 1500, 80))
    mask = np.full((1500,), -1.0, dtype=np.float32)
    want, want_w = O.flash(q, k, v, mask)
    got, got_w = run_gpu(q, k, v, mask)
    assert_close(got, want, 1e-4, 1e-4, what="flash split all masked out")
    assert_close(got_w, want_w, 1e-5, 1e-4, what="flash split all masked weights")
