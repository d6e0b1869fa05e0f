"""Key ranges that begin before a row's first key, end past its last one, are empty the other way round, or have the
type's lowest and highest values for ends: a query sees the keys of [start, end) that there are, in the forward and in
every backward.  Against the oracle, in the bounds of the other direct calls; one row has nothing but such ranges."""

import numpy as np
import pytest
import torch

from tests.test_attention_direct_gpu import GRAD_TOL, LSE_TOL, OUT_TOL, _check_direct, _paged_rows, _run_direct

pytestmark = pytest.mark.gpu

LOW, HIGH = -(2 ** 31), 2 ** 31 - 1
# (with keys, without, in turn)
ODD = [(LOW, 70), (5, LOW), (-1000, 130), (HIGH, HIGH), (LOW, HIGH), (HIGH, LOW), (-64, 64), (LOW, LOW), (100, HIGH), (-5, -2),
       (-1, 1), (300, 200), (-65, 63), (LOW, 0), (0, HIGH), (0, LOW), (127, 129), (LOW, -1), (-HIGH, 192), (10000, HIGH)]


def _ranges(rng, nq, n_keys, n_ranges, every):
    r = np.zeros((n_ranges, 2, nq), dtype=np.int64)
    for i in range(n_ranges):
        r[i, 0] = rng.integers(0, n_keys, size=nq)
        r[i, 1] = r[i, 0] + rng.integers(0, n_keys, size=nq)
        odd = np.arange(i, nq, every)
        r[i, :, odd] = [ODD[(7 * i + j) % len(ODD)] for j in range(len(odd))]
    return r.astype(np.int32)


@pytest.mark.parametrize("mode", [0, 1, 2])  # recomputing, one pass, dS kept
@pytest.mark.parametrize("n_ranges", [1, 2])
@pytest.mark.parametrize("d,hq,hkv", [(128, 4, 2), (64, 2, 2)])
def test_ranges_at_the_limits(gpu, d, hq, hkv, n_ranges, mode):
    from dcp_amd import _lib

    rng, bs = np.random.default_rng(11), 128
    rows = [(nq, nblk, _ranges(rng, nq, nblk * bs, n_ranges, every)) for nq, nblk, every in ((128, 3, 7), (70, 2, 3), (128, 4, 1), (33, 1, 2))]
    pr = _paged_rows(gpu, rows, bs, hq, hkv, d, seed=6)
    before = _lib.load().dcp_attn_bwd_select(mode)
    try:
        worst = _check_direct(pr, _run_direct(pr))
    finally:
        _lib.load().dcp_attn_bwd_select(before)
    assert worst["out"] <= OUT_TOL and worst["lse"] <= LSE_TOL and worst["dq"] <= GRAD_TOL and worst["dkv"] <= GRAD_TOL, worst
