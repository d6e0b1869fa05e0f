"""Forward launches whose rows are split along their keys: the split covers every row's keys once and fits
its rule (CPU); results against dense attention and against the unsplit launch, with parts of one tile,
parts without a visible key, one and two ranges, ragged blocks, and several launches of a plan (GPU)."""

import numpy as np
import pytest
import torch

from dcp_amd.runtime.flash_attention import fwd_parts
from tests.plan_cases import check_against_truth, dense_truth, make_case, run_executor
from tests.test_dkv_groups import PLANS


def test_every_part_of_every_row_once(monkeypatch):
    seqlens = [64, 65, 640, 1000, 2048, 1]
    for share in (1, 3, 8):
        monkeypatch.setattr(fwd_parts, "share_of_a_part", lambda *a: share)
        parts, splits, n_partials = fwd_parts.split_rows(seqlens, 16, 512)
        seen = sorted(map(tuple, parts[:, :3].tolist()))
        counts = [max(1, -(-(-(-n // 64)) // share)) for n in seqlens]
        assert seen == [(row, i, n) for row, n in enumerate(counts) for i in range(n)]
        assert sorted(f + i for _, i, n, f in parts.tolist() if n > 1) == list(range(n_partials))
        assert splits.tolist() == [[r, n, next(f for row, _, _, f in parts.tolist() if row == r), 0] for r, n in enumerate(counts) if n > 1]


def test_rule():
    """Only where the longest row outlasts the rest, and then so that all parts are on the device at once."""
    share = fwd_parts.share_of_a_part
    assert share([], 16, 512) is None
    assert share([11, 6, 4], 16, 512) is None  # too short to be worth the sums
    assert share([64] * 64, 16, 512) is None  # even, and more items than slots
    assert share([256, 240] + [200] * 500, 4, 512) is None
    for tiles, items in (([128], 8), ([32, 28, 24, 20, 16, 12, 8, 4], 16), (list(range(4, 132, 4)), 8)):
        s = share(tiles, items, 512)
        assert s >= fwd_parts.MIN_SHARE and sum(-(-t // s) for t in tiles) * items <= 512
    assert share([400] + [8] * 600, 4, 512) == -(-(400 + 8 * 600) * 4 // 512)


@pytest.mark.gpu
@pytest.mark.parametrize("share", [1, 2, 5])
@pytest.mark.parametrize("name", list(PLANS))
def test_split_forward_matches_dense_attention(gpu, monkeypatch, name, share):
    case = make_case(**PLANS[name])
    whole, _ = run_executor(case, backward=False)
    monkeypatch.setattr(fwd_parts, "share_of_a_part", lambda *a: share)
    split, ex = run_executor(case, backward=False, poison=200.0)
    monkeypatch.setenv("DCP_DIRECT_LOCAL", "0")
    as_written, _ = run_executor(case, backward=False)
    assert ex._fwd_partials is not None
    check_against_truth(split, dense_truth(case, backward=False))
    assert torch.equal(split[0], as_written[0])
    monkeypatch.delenv("DCP_DIRECT_LOCAL")
    replayed, _ = run_executor(case, backward=False, use_graph=True)
    assert torch.equal(split[0], replayed[0]) and torch.equal(split[1], replayed[1])
    # the merged LSE of two launches goes through the merge kernel as written and directly
    np.testing.assert_allclose(split[1].float().cpu().numpy(), whole[1].float().cpu().numpy(), rtol=2e-6, atol=2e-6)
