"""Which dK/dV replicas the backward kernel adds itself (``dkv_groups.analyse``): every (row, kv block)
of a launch in exactly one group, a group's rows attend to one kv block, and group results plus what
the sums still read are the replicas the plan adds, each exactly once (CPU).  On the GPU: grouped
launches against dense attention and against the plan's own replicas, at group sizes from one row to
more than the kernel takes at once."""

from collections import Counter

import pytest
import torch

from dcp_amd.core.instructions import (
    AttnBackwardInstr,
    BufferBlock,
    BufferType,
    CommLaunchInstr,
    CommOp,
    CommType,
    MemcpyInstr,
    SumInstr,
    SumOp,
)
from dcp_amd.runtime.flash_attention import dkv_groups
from dcp_amd.runtime.flash_attention.direct import DirectPlan, analyse as analyse_direct
from tests.plan_cases import check_against_truth, dense_truth, make_case, make_multi_case, run_executor, run_multi_executor, scaled_err

PLANS = {
    # blocks with 1 to 9 rows, several q head blocks per kv head; ragged last blocks
    "causal_gqa": dict(seqlens=[1100, 300, 1, 129], block_size=128, n_heads=8, n_groups=2, head_dim=128, head_block=2, qkv_scale=0.5),
    # two partials per row: one backward launch per partial, one sum over both
    "split": dict(seqlens=[900, 130], block_size=128, n_heads=4, n_groups=2, head_dim=64, head_block=1, n_kv_groups=2,
                  kv_split="contiguous", qkv_scale=0.5),
    # two ranges per query: key tiles of the sink block that most rows do not see (visits without a step)
    "lambda": dict(seqlens=[1500, 130], block_size=256, n_heads=4, n_groups=1, head_dim=128, head_block=2, mask="lambda",
                   mask_kwargs=dict(n_starting=16, l_pretrain=300), qkv_scale=0.5),
    # no grouped queries: a visit of one head's tiles
    "mha_fp16": dict(seqlens=[1300, 70], block_size=128, n_heads=3, n_groups=3, head_dim=64, head_block=3, dtype="fp16", qkv_scale=0.5),
    # 41 rows for the first block: more than a group holds
    "many_rows": dict(seqlens=[41 * 128 - 5], block_size=128, n_heads=2, n_groups=2, head_dim=128, head_block=2, qkv_scale=0.5),
}


def _check_groups(plan, found):
    """Every (row, kv block) pair of a grouped launch is in exactly one group; and, walking the plan once as
    written and once with the groups: whatever reads a dK/dV slot other than a sum finds in it what the plan
    put there, and every sum adds the same replicas (or is left out where its replicas went together)."""
    instrs = plan.instructions
    as_written, with_groups = {}, {}  # slot -> the (instr, row, pos) replicas or other writes added up in it
    local = []  # what groups put into LOCAL_dKV

    def put(block, what):
        if block.buffer_type == BufferType.BUFFER_dKV:
            as_written[block.index] = with_groups[block.index] = Counter([what])

    def same(block):
        if block.buffer_type == BufferType.BUFFER_dKV:
            assert with_groups.get(block.index) == as_written.get(block.index)

    def total(slots, blocks):
        blocks = [b for b in blocks if b.buffer_type == BufferType.BUFFER_dKV]
        assert all(b.index in slots for b in blocks)
        return sum((slots[b.index] for b in blocks), Counter())

    for idx, instr in enumerate(instrs):
        if isinstance(instr, AttnBackwardInstr):
            pairs = {(r, p): slot for r, row in enumerate(instr.dkv_block_table) for p, slot in enumerate(row)}
            for (r, p), slot in pairs.items():
                put(slot, (idx, r, p))
            if idx not in found.groups:
                continue
            for slot in pairs.values():  # (the launch writes the groups' slots only)
                with_groups.pop(slot.index, None)
            groups = found.groups[idx]
            assert sorted(v for g in groups for v in g.visits) == sorted(pairs)
            assert [len(g.visits) for g in groups] == sorted((len(g.visits) for g in groups), reverse=True)
            for g in groups:
                assert 1 <= len(g.visits) <= dkv_groups.MAX_VISITS
                assert len({instr.kv_block_table[r][p].index for r, p in g.visits}) == 1
                added = Counter((idx, r, p) for r, p in g.visits)
                if g.dst.buffer_type == BufferType.BUFFER_dKV:
                    assert g.dst.index == pairs[g.visits[0]].index
                    with_groups[g.dst.index] = added
                else:
                    local.append(added)
        elif isinstance(instr, SumInstr):
            for pos, op in enumerate(instr.ops):
                want = total(as_written, op.src_buffers) if op.src_buffers[0].buffer_type == BufferType.BUFFER_dKV else Counter()
                if pos in found.skip_ops.get(idx, ()):
                    assert want in local
                else:
                    assert total(with_groups, found.sources.get(idx, {}).get(pos, op.src_buffers)) == want
            for pos, op in enumerate(instr.ops):
                put(op.dst_buffer, ("sum", idx, pos))
        elif isinstance(instr, MemcpyInstr):
            for pos, (src, dst) in enumerate(instr.src_dst_pairs):
                same(src)
                put(dst, ("copy", idx, pos))
        elif isinstance(instr, CommLaunchInstr):
            for pos, op in enumerate(instr.comm_ops):
                if op.comm_type == CommType.SEND:
                    same(op.buffer_block)
                else:
                    put(op.buffer_block, ("received", idx, pos))


@pytest.mark.parametrize("limit", [1, 3, 32])
@pytest.mark.parametrize("direct", [False, True])
@pytest.mark.parametrize("name", list(PLANS))
def test_every_replica_is_added_once(monkeypatch, name, direct, limit):
    monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: limit)
    plan = make_case(**PLANS[name])["bw"]
    d = analyse_direct(plan) if direct else DirectPlan()
    found = dkv_groups.analyse(plan, d, 1, 1, 512)
    _check_groups(plan, found)
    if limit == 1:
        assert not found.groups
    else:
        assert any(len(g.visits) > 1 for gs in found.groups.values() for g in gs)


@pytest.mark.parametrize("limit", [2, 32])
@pytest.mark.parametrize("n_stages", [None, 2])
def test_every_replica_of_a_device_is_added_once(monkeypatch, n_stages, limit):
    """Plans with an exchange: sums over replicas and blocks that were received, slots used again."""
    monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: limit)
    case = make_multi_case(n_nodes=1, n_devices_per_node=2, seqlens=[700, 330], block_size=128, n_heads=4, n_groups=2, head_dim=64,
                           head_block=2, n_stages=n_stages)
    for plan in case["bw"]:
        found = dkv_groups.analyse(plan, DirectPlan(), 1, 1, 512)
        _check_groups(plan, found)
        assert any(len(g.visits) > 1 for gs in found.groups.values() for g in gs)


@pytest.mark.parametrize("how", ["sent", "copied", "added_twice", "received"])
def test_replicas_with_another_reader_are_left_alone(monkeypatch, how):
    """A replica that is sent to another device, copied, added by a second sum, or whose slot a received block
    takes, keeps a group and a slot of its own, and the sum still adds that slot."""
    monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: 32)
    plan = make_case(**PLANS["causal_gqa"])["bw"]
    at = next(i for i, instr in enumerate(plan.instructions) if isinstance(instr, AttnBackwardInstr))
    group = next(g for g in dkv_groups.analyse(plan, analyse_direct(plan), 1, 1, 512).groups[at] if len(g.visits) > 3)
    row, pos = group.visits[2]
    slot = plan.instructions[at].dkv_block_table[row][pos]
    elsewhere = BufferBlock(BufferType.BUFFER_dKV, 10 ** 6, slot.n_tokens)
    plan.instructions.insert(at + 1, {
        "sent": lambda: CommLaunchInstr("k", [CommOp(CommType.SEND, (0, 1), slot)], None),
        "received": lambda: CommLaunchInstr("k", [CommOp(CommType.RECV, (0, 1), slot)], None),
        "copied": lambda: MemcpyInstr([(slot, elsewhere)]),
        "added_twice": lambda: SumInstr([SumOp([slot], elsewhere)], False),
    }[how]())
    found = dkv_groups.analyse(plan, analyse_direct(plan), 1, 1, 512)
    _check_groups(plan, found)
    (alone,) = [g for g in found.groups[at] if (row, pos) in g.visits]
    assert alone.visits == [(row, pos)] and alone.dst == slot
    adding = [(j, k) for j, i in enumerate(plan.instructions) if j > at + 1 and isinstance(i, SumInstr) for k, op in enumerate(i.ops)
              if slot in op.src_buffers]
    assert adding
    for j, k in adding:
        assert k not in found.skip_ops.get(j, ()) and slot in found.sources.get(j, {}).get(k, plan.instructions[j].ops[k].src_buffers)


def _without_keys_of_a_row(plan):
    """Leaves a row of the backward plan (the first of one kv block) nothing to attend to, and takes its
    replica from the sum.  The slots that are gone."""
    gone = set()
    for instr in plan.instructions:
        if isinstance(instr, AttnBackwardInstr):
            row = next(r for r, blocks in enumerate(instr.kv_block_table) if len(blocks) == 1)
            gone.update(b.index for b in instr.dkv_block_table[row])
            instr.kv_block_table[row], instr.dkv_block_table[row], instr.seqlens_kv[row] = [], [], 0
        elif isinstance(instr, SumInstr):
            for op in instr.ops:
                if op.src_buffers[0].buffer_type == BufferType.BUFFER_dKV and len(op.src_buffers) > 1:
                    op.src_buffers = [b for b in op.src_buffers if b.index not in gone]
    return gone


@pytest.mark.parametrize("limit", [3, 32])
def test_a_row_without_kv_blocks(monkeypatch, limit):
    monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: limit)
    plan = make_case(**PLANS["causal_gqa"])["bw"]
    assert _without_keys_of_a_row(plan)
    found = dkv_groups.analyse(plan, analyse_direct(plan), 1, 1, 512)
    assert found.groups
    _check_groups(plan, found)


def _executor_without_a_device(monkeypatch, plan, run=None, prep=None):
    """An executor that can be asked for its groups on a machine without a GPU; ``run`` and ``prep``: handlers
    that take the place of this package's, by instruction type."""
    from types import SimpleNamespace

    from dcp_amd.core.executor import HandlerTable
    from dcp_amd.runtime.flash_attention import executor as module

    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda d: SimpleNamespace(multi_processor_count=256))
    ex = module.AttentionExecutor.__new__(module.AttentionExecutor)
    ex.fabric, ex.execution_plan, ex._direct, ex.dkv_groups = None, plan, DirectPlan(), True
    ex.buffer_per_token_shape = {t: info.per_token_shape for t, info in plan.buffer_info.items()}
    ex._handlers, ex._prep_handlers = HandlerTable("run"), HandlerTable("prep")
    for kind, name in ((AttnBackwardInstr, "attn_bw"), (SumInstr, "sum")):
        ex._handlers.register(kind, (run or {}).get(kind, getattr(module, f"_handle_{name}")))
        ex._prep_handlers.register(kind, (prep or {}).get(kind, getattr(module, f"_prepare_{name}")))
    return ex


@pytest.mark.parametrize("table", ["run", "prep"])
@pytest.mark.parametrize("kind", [AttnBackwardInstr, SumInstr])
def test_no_groups_where_a_handler_is_the_callers_own(monkeypatch, table, kind):
    """The plug-in surface: an own handler writes and adds every replica, as the plan says."""
    plan = make_case(**PLANS["causal_gqa"])["bw"]
    monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: 32)
    assert _executor_without_a_device(monkeypatch, plan)._group_dkv_replicas().groups
    own = {kind: lambda e, i: None}
    assert _executor_without_a_device(monkeypatch, plan, **{table: own})._group_dkv_replicas() == dkv_groups.DkvGroups()
    ex = _executor_without_a_device(monkeypatch, plan)
    monkeypatch.setattr(ex, "_execute_instruction", lambda instr: None)  # (runs them in its own way)
    assert ex._group_dkv_replicas() == dkv_groups.DkvGroups()


def test_groups_can_be_turned_off(monkeypatch):
    monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: 32)
    ex = _executor_without_a_device(monkeypatch, make_case(**PLANS["causal_gqa"])["bw"])
    ex.dkv_groups = False
    assert ex._group_dkv_replicas() == dkv_groups.DkvGroups()


def test_no_groups_in_plans_without_a_backward_or_its_tensor(monkeypatch):
    """Plans that have dK/dV slots but no backward launch (and no dQ), or no LOCAL_dKV."""
    monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: 32)
    sums = make_case(**PLANS["causal_gqa"])["bw"]
    sums.instructions = [i for i in sums.instructions if isinstance(i, SumInstr)]
    del sums.buffer_info[BufferType.BUFFER_dQ]
    assert _executor_without_a_device(monkeypatch, sums)._group_dkv_replicas() == dkv_groups.DkvGroups()
    slots_only = make_case(**PLANS["causal_gqa"])["bw"]
    del slots_only.buffer_info[BufferType.LOCAL_dKV]
    assert _executor_without_a_device(monkeypatch, slots_only)._group_dkv_replicas() == dkv_groups.DkvGroups()


@pytest.mark.parametrize("how", ["written", "read"])
def test_a_local_block_named_twice_is_left_to_its_sums(monkeypatch, how):
    """The launch writes LOCAL_dKV earlier than the sum would: not if the plan does anything else with the
    block, here between the two."""
    monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: 32)

    def local_blocks(plan):
        found = dkv_groups.analyse(plan, analyse_direct(plan), 1, 1, 512)
        _check_groups(plan, found)
        return {g.dst.index: g.dst for gs in found.groups.values() for g in gs if g.dst.buffer_type == BufferType.LOCAL_dKV}

    plan = make_case(**PLANS["causal_gqa"])["bw"]
    before = local_blocks(plan)
    block = next(iter(before.values()))
    slot = BufferBlock(BufferType.BUFFER_KV, 10 ** 6, block.n_tokens)
    between = next(i for i, instr in enumerate(plan.instructions) if isinstance(instr, AttnBackwardInstr)) + 1
    plan.instructions.insert(between, SumInstr([SumOp([slot], block)], True) if how == "written" else MemcpyInstr([(block, slot)]))
    assert set(local_blocks(plan)) == set(before) - {block.index}


@pytest.mark.parametrize("parts", [(1, 1), (2, 1)])
def test_a_plan_with_an_unknown_instruction_is_left_alone(monkeypatch, parts):
    """An instruction of a kind the analysis does not know may read any replica."""
    monkeypatch.setattr(dkv_groups, "parts_per_visit", lambda *a: parts)
    monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: 1 if parts != (1, 1) else 32)
    plan = make_case(**PLANS["causal_gqa"])["bw"]
    assert dkv_groups.analyse(plan, DirectPlan(), 1, 1, 512, 2).groups
    for at in (0, len(plan.instructions) // 2, len(plan.instructions)):
        other = make_case(**PLANS["causal_gqa"])["bw"]
        other.instructions.insert(at, object())
        assert dkv_groups.analyse(other, DirectPlan(), 1, 1, 512, 2) == dkv_groups.DkvGroups()


@pytest.mark.parametrize("parts", [(1, 2), (2, 1), (3, 4)])
@pytest.mark.parametrize("name", ["causal_gqa", "split", "lambda"])
def test_parts_cover_every_head_and_tile_once(monkeypatch, name, parts):
    """A plan whose pairs are split: each pair's parts cover the q heads of its kv head and the 64-query
    tiles exactly once, every partial is added by exactly one sum, the one that adds the replica."""
    monkeypatch.setattr(dkv_groups, "parts_per_visit", lambda *a: parts)
    kw = PLANS[name]
    plan, bs = make_case(**kw)["bw"], kw["block_size"]
    n_heads, n_tiles = 5, bs // 64
    found = dkv_groups.analyse(plan, analyse_direct(plan), 1, bs // 128, 512, n_heads)
    added = [p for ops in found.partials.values() for op in ops.values() for p in op]
    assert sorted(added) == list(range(found.n_partials))
    for idx, groups in found.groups.items():
        instr = plan.instructions[idx]
        seen, of_pair = {}, {}
        for g in groups:
            (pair,) = g.visits
            assert isinstance(g.dst, int)
            heads = range(*g.heads) if g.heads != (0, 0) else range(n_heads)
            n, i = g.tiles
            cells = [(h, t) for h in heads for t in range(n_tiles) if n == 0 or t % n == i]
            assert not set(cells) & seen.setdefault(pair, set())
            seen[pair].update(cells)
            of_pair.setdefault(pair, []).append(g.dst)
        assert set(seen) == {(r, p) for r, row in enumerate(instr.kv_block_table) for p in range(len(row))}
        assert all(len(cells) == n_heads * n_tiles for cells in seen.values())
        for (row, pos), partials in of_pair.items():
            slot = instr.dkv_block_table[row][pos].index
            (op,) = [(j, k) for j, i in enumerate(plan.instructions) if isinstance(i, SumInstr)
                     for k, o in enumerate(i.ops) if any(b.buffer_type == BufferType.BUFFER_dKV and b.index == slot for b in o.src_buffers)
                     and k in found.partials.get(j, {})]
            assert set(partials) <= set(found.partials[op[0]][op[1]])


def test_group_size_rule():
    """One row per group where the launch does not fill the device once, more the more often it does, never more
    than the kernel takes."""
    assert dkv_groups.visits_per_group(60, 8, 512) == 1
    assert dkv_groups.visits_per_group(10 ** 6, 8, 512) == dkv_groups.MAX_VISITS
    assert 1 < dkv_groups.visits_per_group(2544, 8, 512) < dkv_groups.MAX_VISITS
    # and parts of a row only where the rows are fewer than half the device's workgroups
    assert dkv_groups.parts_per_visit(6, 4, 512, 4, 8) == (4, 2)
    assert dkv_groups.parts_per_visit(24, 8, 512, 5, 16) == (2, 1)
    assert dkv_groups.parts_per_visit(40, 8, 512, 5, 16) == (1, 1)
    assert dkv_groups.parts_per_visit(1, 2, 512, 1, 4) == (1, 1)


@pytest.mark.parametrize("pairs,rows", [(0.99, 1), (1.19, 2), (2.38, 3), (3.12, 3), (3.53, 4), (7.75, 8), (8.1, 8), (15.9, 8), (25, 13), (80, 32)])
def test_rows_per_group_by_pairs_per_slot(pairs, rows):
    assert dkv_groups.visits_per_group(round(pairs * 512), 1, 512) == rows


@pytest.mark.gpu
@pytest.mark.parametrize("limit", [2, 32])
@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("name", list(PLANS))
def test_grouped_backward_matches_dense_attention(gpu, monkeypatch, name, mode, limit):
    from dcp_amd import _lib

    lib = _lib.load()
    case = make_case(**PLANS[name])
    before = lib.dcp_attn_bwd_select(mode)
    try:
        monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: 1)
        single, _ = run_executor(case, backward=True)
        monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: limit)
        grouped, ex = run_executor(case, backward=True, poison=200.0)
        monkeypatch.setenv("DCP_DIRECT_LOCAL", "0")
        as_written, _ = run_executor(case, backward=True)
    finally:
        lib.dcp_attn_bwd_select(before)
    assert any(len(g.visits) == min(limit, 2) or len(g.visits) > 2 for gs in ex._dkv_groups.groups.values() for g in gs)
    check_against_truth(grouped, dense_truth(case, backward=True))
    same_dq = torch.equal(grouped[2], single[2])  # dQ does not depend on the grouping
    same_as_written = torch.equal(grouped[3], as_written[3]) and torch.equal(grouped[2], as_written[2])
    assert same_dq and same_as_written


@pytest.mark.gpu
@pytest.mark.parametrize("parts", [(1, 1), (1, 2), (2, 1), (2, 3)])
@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("name", ["causal_gqa", "split", "lambda", "mha_fp16"])
def test_backward_in_parts_matches_dense_attention(gpu, monkeypatch, name, mode, parts):
    """Parts without a single visible key, of one head, of every third tile; two launches that add to one sum."""
    from dcp_amd import _lib

    monkeypatch.setattr(dkv_groups, "parts_per_visit", lambda *a: (min(parts[0], a[3]), min(parts[1], a[4])))
    monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: 1)
    lib = _lib.load()
    case = make_case(**PLANS[name])
    before = lib.dcp_attn_bwd_select(mode)
    try:
        direct, ex = run_executor(case, backward=True, poison=200.0)
        monkeypatch.setenv("DCP_DIRECT_LOCAL", "0")
        as_written, _ = run_executor(case, backward=True)
    finally:
        lib.dcp_attn_bwd_select(before)
    split = parts[1] > 1 or parts[0] > 1 and name in ("causal_gqa", "lambda")  # (the others have one q head per kv head in a block)
    assert (ex._dkv_groups.n_partials > 0) == split
    check_against_truth(direct, dense_truth(case, backward=True))
    same = torch.equal(direct[3], as_written[3]) and torch.equal(direct[2], as_written[2])
    assert same


@pytest.mark.gpu
def test_grouped_backward_with_an_exchange(gpu, monkeypatch):
    case = make_multi_case(n_nodes=1, n_devices_per_node=2, seqlens=[700, 330], block_size=128, n_heads=4, n_groups=2, head_dim=128,
                           head_block=2, n_stages=2)
    single, _ = run_multi_executor(case, backward=True)
    monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: 32)
    grouped, _ = run_multi_executor(case, backward=True, repeats=2)
    # unscaled inputs and partials that cross the exchange rounded: the bound of the exchange tests
    err = scaled_err(grouped[3].float().numpy(), dense_truth(case, backward=True)[3])
    same_dq = torch.equal(grouped[2], single[2])
    assert same_dq and err <= 4e-2


def _with_exact_key_counts(case):
    """The case's backward plan with the rows' key counts taken from their blocks' tokens: a row whose last
    block is ragged ends inside it.  How many rows that are."""
    n = 0
    for instr in case["bw"].instructions:
        if isinstance(instr, AttnBackwardInstr):
            exact = [sum(block.n_tokens for block in row) for row in instr.kv_block_table]
            n += sum(a != b for a, b in zip(exact, instr.seqlens_kv))
            instr.seqlens_kv = exact
    return n


@pytest.mark.gpu
@pytest.mark.parametrize("limit", [1, 2, 32])
@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("name", ["causal_gqa", "split", "lambda"])
def test_rows_that_end_inside_a_block(gpu, monkeypatch, name, mode, limit):
    """Key counts that are no multiples of the block size, nor of the 64 keys of a dS piece: the masked keys of
    whole blocks contribute exact zeros, so the results are those of whole blocks bit for bit.  The
    backward's scratch holds NaNs before."""
    from dcp_amd import _lib
    from dcp_amd.runtime.flash_attention.executor import AttentionExecutor

    prepare = AttentionExecutor.prepare

    def with_nans_in_scratch(self, forward=True):
        prepare(self, forward)
        if self._bwd_workspace is not None:
            self._bwd_workspace.fill_(255)

    monkeypatch.setattr(AttentionExecutor, "prepare", with_nans_in_scratch)
    monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: limit)
    monkeypatch.setattr(dkv_groups, "parts_per_visit", lambda *a: (1, 1))
    lib = _lib.load()
    case = make_case(**PLANS[name])
    before = lib.dcp_attn_bwd_select(mode)
    try:
        whole, _ = run_executor(case, backward=True)
        assert _with_exact_key_counts(case) > 0
        exact, ex = run_executor(case, backward=True, poison=200.0)
    finally:
        lib.dcp_attn_bwd_select(before)
    assert bool(ex._dkv_groups.groups) == (limit > 1)
    check_against_truth(exact, dense_truth(case, backward=True))
    same_dq, same_dkv = torch.equal(exact[2], whole[2]), torch.equal(exact[3], whole[3])
    assert same_dq and same_dkv


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [0, 2])
def test_grouped_backward_of_a_row_without_kv_blocks(gpu, monkeypatch, mode):
    from dcp_amd import _lib

    lib = _lib.load()
    case = make_case(**PLANS["causal_gqa"])
    assert _without_keys_of_a_row(case["bw"])
    monkeypatch.setattr(dkv_groups, "parts_per_visit", lambda *a: (1, 1))
    before = lib.dcp_attn_bwd_select(mode)
    try:
        monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: 1)
        single, _ = run_executor(case, backward=True)
        monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: 32)
        grouped, ex = run_executor(case, backward=True, poison=200.0)
    finally:
        lib.dcp_attn_bwd_select(before)
    assert ex._dkv_groups.groups
    same_dq = torch.equal(grouped[2], single[2])
    # nine replicas of about one, each rounded to bf16 (2^-9) before the plan's own sum adds them
    assert same_dq and scaled_err(grouped[3].float().numpy(), single[3].float().numpy()) <= 2e-2


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [AttnBackwardInstr, SumInstr])
def test_handlers_of_the_callers_own_find_every_replica(gpu, monkeypatch, kind):
    """A caller's own backward that writes the replicas, and a caller's own sum that reads them."""
    from dcp_amd.runtime.flash_attention import executor as module

    case = make_case(**PLANS["causal_gqa"])
    with monkeypatch.context() as m:
        m.setattr(dkv_groups, "visits_per_group", lambda *a: 1)
        m.setattr(dkv_groups, "parts_per_visit", lambda *a: (1, 1))
        want, _ = run_executor(case, backward=True)
    monkeypatch.setattr(dkv_groups, "visits_per_group", lambda *a: 32)
    theirs = {AttnBackwardInstr: module._handle_attn_bw, SumInstr: module._handle_sum}[kind]
    seen = []

    def own(ex, instr):
        seen.append(ex.instr_index)
        if kind is AttnBackwardInstr:
            theirs(ex, instr)
            return
        cu, bs = ex.execution_plan.local_cu_seqlens, ex.buffer_block_sizes
        for op in instr.ops:  # the plan's sum in torch: added in fp32 in the plan's order, rounded once
            n, dst = op.dst_buffer.n_tokens, op.dst_buffer
            total = sum(ex.buffers[b.buffer_type].view(-1, bs[b.buffer_type], *ex.buffer_per_token_shape[b.buffer_type])[b.index, :n].float()
                        for b in op.src_buffers)
            to = ex.buffers[dst.buffer_type]
            if instr.output_is_unpadded:
                to[cu[dst.index] : cu[dst.index] + n] = total.to(to.dtype)
            else:
                to.view(-1, bs[dst.buffer_type], *ex.buffer_per_token_shape[dst.buffer_type])[dst.index, :n] = total.to(to.dtype)

    monkeypatch.setattr(module, "get_executor", _with_own_handler(module.get_executor, kind, own))
    monkeypatch.setenv("DCP_DIRECT_LOCAL", "0")  # (its sums may leave out scatters, which an own handler makes)
    got, ex = run_executor(case, backward=True)
    assert seen and not ex._dkv_groups.groups
    assert torch.equal(got[2], want[2]) and torch.equal(got[3], want[3])


def _with_own_handler(get_executor, kind, own):
    def make(*args, **kw):
        ex = get_executor(*args, **kw)
        ex._handlers._by_type[kind] = own
        return ex

    return make


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(PLANS))
def test_plan_as_written(gpu, monkeypatch, name):
    """Without groups dK/dV are the sums of the rounded replicas the plan asks for, whether or not copies
    are left out, and every replica is in its slot."""
    from collections import defaultdict

    case = make_case(**PLANS[name])
    grouped, _ = run_executor(case, backward=True)
    monkeypatch.setenv("DCP_DKV_GROUPS", "0")
    direct, ex = run_executor(case, backward=True)
    assert not ex.dkv_groups and not ex._dkv_groups.groups
    monkeypatch.setenv("DCP_DIRECT_LOCAL", "0")
    as_written, ex = run_executor(case, backward=True, poison=200.0)
    assert torch.equal(direct[2], as_written[2]) and torch.equal(direct[3], as_written[3])
    assert torch.equal(grouped[2], as_written[2])  # (dQ does not depend on the grouping)
    assert scaled_err(grouped[3].float().numpy(), as_written[3].float().numpy()) <= 2e-2
    cu, slots, written = case["bw"].local_cu_seqlens, ex.buffers["BufferdKV"], defaultdict(int)
    for instr in case["bw"].instructions:
        if isinstance(instr, AttnBackwardInstr):
            for row in instr.dkv_block_table:
                for block in row:
                    written[block.index] += 1
        for op in instr.ops if isinstance(instr, SumInstr) else []:
            src, dst = op.src_buffers, op.dst_buffer
            if dst.buffer_type != BufferType.LOCAL_dKV or not all(written[b.index] == 1 for b in src):
                continue
            total = sum(slots[b.index, : dst.n_tokens].float() for b in src)
            got = ex.buffers["LocaldKV"][cu[dst.index] : cu[dst.index] + dst.n_tokens]
            assert torch.equal(got, total.to(got.dtype))
