"""Forward launches from a table of their work items: the table names every 128 queries of every row (or part of a row)
once and keeps a row's on one XCD (CPU); results are those of the launch that counts the items itself (GPU)."""

from math import gcd

import numpy as np
import pytest
import torch

from dcp_amd.core.instructions import AttnInstr
from dcp_amd.runtime.flash_attention import executor, fwd_parts, items
from tests.plan_cases import check_against_truth, dense_truth, make_case, run_executor
from tests.test_attention_direct_gpu import _paged_rows
from tests.test_dkv_groups import PLANS


@pytest.mark.parametrize("n_kv_heads", [1, 2, 3, 8])
@pytest.mark.parametrize("seqlens_q", [[1], [128, 129, 127, 1, 1024, 300] * 7, [5, 0, 260], list(range(1, 40))])
def test_every_tile_once(seqlens_q, n_kv_heads):
    rng = np.random.default_rng(0)
    seqlens_kv = rng.integers(1, 4000, size=len(seqlens_q)).tolist()
    table = items.forward_items(seqlens_q, seqlens_kv, n_kv_heads)
    want = [(row, t, 65536, 0) for row, n in enumerate(seqlens_q) for t in range(-(-n // 128))]
    assert sorted(map(tuple, table.tolist())) == want
    # positions that come round to one XCD hold whole rows, until the first XCD's are out (three rounds at least, here)
    lanes = 8 // gcd(8, n_kv_heads)
    xcds = {}
    for at, (row, *_) in enumerate(table[: 3 * lanes].tolist()):
        xcds.setdefault(row, set()).add(at % lanes)
    assert len(seqlens_q) < 39 or all(len(x) == 1 for x in xcds.values())


def test_parts_of_rows():
    seqlens_q, seqlens_kv = [300, 128, 64, 512], [4096, 640, 64, 2048]
    parts = np.asarray([[0, 0, 2, 0], [0, 1, 2, 0], [3, 0, 1, 0], [1, 0, 1, 0], [2, 0, 1, 0]], dtype=np.int32)
    table = items.forward_items(seqlens_q, seqlens_kv, 8, parts=parts)
    want = [(row, t, i + (n << 16), f) for row, i, n, f in parts.tolist() for t in range(-(-seqlens_q[row] // 128))]
    assert sorted(map(tuple, table.tolist())) == sorted(want)


def test_rule():
    pays = lambda seqlens, block_size, n_heads=32, n_slots=100: items.pays(seqlens, block_size, n_heads, n_slots)
    assert not pays([], 1024) and not pays([0], 1024)
    assert pays([290] * 9, 1024) and not pays([1000] * 9, 1024) and not pays([256] * 9, 256) and pays([100] * 9, 256)
    assert not pays([290] * 9, 1024, 1) and not pays([290] * 9, 1024, 8, 9 * 8 * 8) and pays([290] * 9, 1024, 8, 9 * 8 * 8 - 1)


def test_rule_of_the_queue():
    each = items.one_workgroup_each
    assert not each([], [], 8, 512) and not each([128] * 64, [640] * 64, 8, 512)  # all at once
    assert each([128] * 65, [640] * 65, 8, 512) and each([100] * 65, [640] * 65, 8, 512)
    assert each([128] * 128, [64 * 32] * 128, 8, 512) and not each([128] * 128, [64 * 32 + 1] * 128, 8, 512)


def _launches(ex, case):
    """The forward launches' parts, items and whether a workgroup is started for each."""
    return [ex._args_cache[i][-4:-1] for i, instr in enumerate(case["fw"].instructions) if isinstance(instr, AttnInstr)]


@pytest.mark.gpu
@pytest.mark.parametrize("share", [None, 2])
@pytest.mark.parametrize("name", list(PLANS))
def test_same_results(gpu, monkeypatch, name, share):
    case = make_case(**PLANS[name])
    if share:
        monkeypatch.setattr(fwd_parts, "share_of_a_part", lambda *a: share)
    monkeypatch.setattr(executor, "items_pay", lambda *a: False)
    counted, ex = run_executor(case, backward=False)
    assert all(items is None for _, items, _ in _launches(ex, case))
    monkeypatch.setattr(executor, "items_pay", lambda *a: True)
    listed, ex = run_executor(case, backward=False, poison=200.0)
    assert all(items is not None for _, items, _ in _launches(ex, case))
    assert share is None or any(parts is not None for parts, _, _ in _launches(ex, case))
    assert torch.equal(counted[0], listed[0]) and torch.equal(counted[1], listed[1])
    check_against_truth(listed, dense_truth(case, backward=False))
    replayed, _ = run_executor(case, backward=False, use_graph=True)
    assert torch.equal(listed[0], replayed[0]) and torch.equal(listed[1], replayed[1])


@pytest.mark.gpu
@pytest.mark.parametrize("listed", [False, True])
@pytest.mark.parametrize("name", list(PLANS))
def test_a_workgroup_each(gpu, monkeypatch, name, listed):
    """More work items than slots, with and without the table: the launch without a queue, the same bits."""
    case = make_case(**dict(PLANS[name], seqlens=PLANS[name]["seqlens"] * 40))
    monkeypatch.setattr(executor, "one_workgroup_each", lambda *a: False)
    monkeypatch.setattr(executor, "items_pay", lambda *a: listed)
    queued, ex = run_executor(case, backward=False)
    slots = 2 * torch.cuda.get_device_properties(gpu).multi_processor_count
    for instr in case["fw"].instructions:
        assert not isinstance(instr, AttnInstr) or sum(-(-row[0].n_tokens // 128) for row in instr.q_block_table) * case["head_block"] > slots
    assert all(parts is None and (items is not None) == listed and not one_each for parts, items, one_each in _launches(ex, case))
    monkeypatch.setattr(executor, "one_workgroup_each", lambda *a: True)
    each, ex = run_executor(case, backward=False, poison=200.0)
    assert all(parts is None and (items is not None) == listed and one_each for parts, items, one_each in _launches(ex, case))
    assert torch.equal(queued[0], each[0]) and torch.equal(queued[1], each[1])
    replayed, _ = run_executor(case, backward=False, use_graph=True)
    assert torch.equal(each[0], replayed[0]) and torch.equal(each[1], replayed[1])


def _rows(gpu):
    """Four rows of up to 300 queries in blocks of 512 and 1 to 3 blocks of keys; four q heads, two kv heads."""
    rng = np.random.default_rng(3)
    rows = [(nq, nblk, np.stack([np.zeros(nq), rng.integers(1, nblk * 512, size=nq)])[None]) for nq, nblk in ((300, 3), (128, 1), (1, 2), (130, 1))]
    return _paged_rows(gpu, rows, 512, 4, 2, 64, seed=2)


def _forward(pr, **options):
    from dcp_amd.flash_attn_interface import _flash_attn_varlen_forward

    q, kv, slots = pr["q"], pr["kv"], pr["slots"]
    out, lse = torch.full_like(q, 3.0), torch.full((q.shape[2], q.shape[0], pr["bs"]), 3.0, device=q.device)
    _flash_attn_varlen_forward(q, kv[:, :, 0], kv[:, :, 1], pr["cu_q"], pr["cu_kv"], pr["total_q"], pr["bs"], pr["max_kv"] * pr["bs"], 0.0,
                               q.shape[-1] ** -0.5, attn_range=pr["rng"], q_block_table=slots, kv_block_table=pr["kv_table"],
                               out_block_table=slots, out_=out, lse_=lse, **options)
    torch.cuda.synchronize()
    return out, lse


@pytest.mark.gpu
@pytest.mark.parametrize("one_each", [False, True])
def test_an_empty_table_is_no_work(gpu, one_each):
    out, lse = _forward(_rows(gpu), items=torch.zeros((0, 4), dtype=torch.int32, device=gpu), one_each=one_each)
    assert (out == 3.0).all() and (lse == 3.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("one_each", [False, True])
def test_the_launch_is_its_table(gpu, one_each):
    """Queries whose 128 are left out of the table are not written, the others are those of a launch without one."""
    pr = _rows(gpu)
    want = _forward(pr, one_each=one_each)
    table = items.forward_items([nq for nq, _, _ in pr["rows"]], [nblk * 512 for _, nblk, _ in pr["rows"]], 2)
    left_out = [(0, 1), (2, 0), (3, 0)]  # (row, which 128 of its queries)
    table = table[[(row, tile) not in left_out for row, tile, _, _ in table.tolist()]]
    got = _forward(pr, items=torch.from_numpy(table).to(gpu), one_each=one_each)
    for row, (nq, _, _) in enumerate(pr["rows"]):
        for tile in range(-(-nq // 128)):
            here = slice(tile * 128, min(tile * 128 + 128, nq))
            written = (want[0][row, here], want[1][:, row, here])
            found = (got[0][row, here], got[1][:, row, here])
            if (row, tile) in left_out:
                assert all((t == 3.0).all() for t in found)
            else:
                assert all(torch.equal(a, b) for a, b in zip(found, written))
