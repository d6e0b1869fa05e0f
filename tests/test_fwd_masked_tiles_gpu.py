"""Forward rows whose ranges end inside key tiles that follow whole ones: those tiles are multiplied without the mask and get
it afterwards, weights are taken against a reference that such a tile may have to raise, and rows that see
nothing ride along in waves of rows that do.  Against the oracle, in the bounds of the other direct calls."""

import numpy as np
import pytest
import torch

from tests.test_attention_direct_gpu import GRAD_TOL, LSE_TOL, OUT_TOL, _check_direct, _paged_rows, _run_direct

pytestmark = pytest.mark.gpu


def _ranges(rng, nq, n_keys, n_ranges, empty):
    """Everybody sees the first 64 keys and a random number more (and a second window); some see nothing."""
    r = np.zeros((n_ranges, 2, nq), dtype=np.int32)
    r[0, 1] = 64 + rng.integers(0, n_keys - 63, size=nq)
    if n_ranges == 2:
        r[1, 0] = rng.integers(0, n_keys, size=nq)
        r[1, 1] = np.minimum(r[1, 0] + rng.integers(0, 150, size=nq), n_keys)
    r[:, :, rng.random(nq) < empty] = 0
    return r


@pytest.mark.parametrize("scale", [1.0, 32.0])  # of the last block's keys: the masked tiles raise the maximum
@pytest.mark.parametrize("empty", [0.0, 0.3])
@pytest.mark.parametrize("n_ranges", [1, 2])
@pytest.mark.parametrize("d,hq,hkv", [(128, 4, 2), (64, 2, 2)])
def test_masked_tiles_after_whole_ones(gpu, d, hq, hkv, n_ranges, empty, scale):
    rng = np.random.default_rng(5)
    bs = 128
    rows = [(nq, nblk, _ranges(rng, nq, nblk * bs, n_ranges, empty)) for nq, nblk in ((128, 3), (70, 2), (33, 4), (1, 2), (97, 1))]
    pr = _paged_rows(gpu, rows, bs, hq, hkv, d, seed=9)
    if scale != 1.0:
        for b, (_, nblk, _) in enumerate(rows):
            slot = int(pr["host"]["kv_table"][b, nblk - 1])
            pr["host"]["kv"][slot, :, 0] *= scale
        pr["kv"] = pr["host"]["kv"].to(gpu)
    worst = _check_direct(pr, _run_direct(pr, backward=scale == 1.0))
    assert worst["out"] <= OUT_TOL and worst["lse"] <= (LSE_TOL if scale == 1.0 else 2e-3)
    if scale == 1.0:
        assert worst["dq"] <= GRAD_TOL and worst["dkv"] <= GRAD_TOL


@pytest.mark.parametrize("n_ranges", [1, 2])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_a_query_that_is_not_finite_keeps_to_itself(gpu, value, n_ranges):
    """The weights of its wave are checked and taken again at every tile; the queries beside it are as accurate as
    ever, and one that sees nothing has out = 0 and lse = +inf whatever its q holds."""
    rng, bs = np.random.default_rng(7), 128
    rows = [(nq, nblk, _ranges(rng, nq, nblk * bs, n_ranges, 0.2)) for nq, nblk in ((128, 3), (70, 2))]
    pr = _paged_rows(gpu, rows, bs, 4, 2, 128, seed=4)
    want = _run_direct(pr, backward=False)
    spoilt = [(b, i) for b, (nq, _, ranges) in enumerate(rows) for i in range(5, nq, 17) if (ranges[:, 1, i] > ranges[:, 0, i]).any()]
    nothing = [(b, i) for b, (nq, _, ranges) in enumerate(rows) for i in range(nq) if not (ranges[:, 1, i] > ranges[:, 0, i]).any()]
    assert spoilt and nothing
    for b, i in spoilt + nothing:
        pr["q"][b, i, :, ::3] = value
    got = _run_direct(pr, backward=False)
    for b, i in nothing:
        assert (got[0][b, i] == 0).all() and np.isposinf(got[1][:, b, i]).all()
    for b, i in spoilt:
        got[0][b, i], got[1][:, b, i] = want[0][b, i], want[1][:, b, i]
    worst = _check_direct(pr, got)
    assert worst["out"] <= OUT_TOL and worst["lse"] <= LSE_TOL
