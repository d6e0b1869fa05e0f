"""The native analyses of a plan (``runtime/flash_attention/native.py``) find what the Python ones find, in plans as
planners make them and in plans changed at random, and leave to them what they do not take (CPU)."""

import copy
import random
import time

import numpy as np
import pytest

from dcp_amd.core.instructions import (
    AttnBackwardInstr,
    AttnInstr,
    AttnReductionInstr,
    BarrierInstr,
    BufferBlock,
    BufferType,
    MemcpyInstr,
    ReductionOp,
    SumInstr,
    SumOp,
)
from dcp_amd.runtime.flash_attention import direct, dkv_groups, executor, native
from tests.plan_cases import make_case

CASES = {
    "causal_gqa": dict(seqlens=[1100, 300, 1, 129], block_size=128, n_heads=8, n_groups=2, head_dim=128, head_block=2),
    "split": dict(seqlens=[900, 130], block_size=128, n_heads=4, n_groups=2, head_dim=64, head_block=1, n_kv_groups=2, kv_split="contiguous"),
    "folded": dict(seqlens=[900, 130], block_size=128, n_heads=4, n_groups=2, head_dim=64, head_block=1, n_kv_groups=3, fold=True),
    "lambda": dict(seqlens=[2500, 130], block_size=128, n_heads=4, n_groups=1, head_dim=128, head_block=2, mask="lambda",
                   mask_kwargs=dict(n_starting=16, l_pretrain=300)),
    "many_rows": dict(seqlens=[41 * 128 - 5], block_size=128, n_heads=2, n_groups=2, head_dim=128, head_block=2),
}


def _plans(name):
    case = make_case(**CASES[name])
    return case["fw"], case["bw"]


def _same_direct(plan):
    found = native.direct(plan.instructions)
    assert found is not None
    assert direct.DirectPlan(*found) == direct._analyse_any(plan)


def _same_groups(plan, limit, analysed):
    limits = {i: limit for i, instr in enumerate(plan.instructions) if isinstance(instr, AttnBackwardInstr)}
    found = native.dkv(plan.instructions, [limits.get(i, 1) for i in range(len(plan.instructions))], analysed.redirect_ops, dkv_groups.Group)
    assert found is not None
    expected = dkv_groups._analyse_any(plan, analysed, limits, {i: (1, 1) for i in limits}, 1)
    assert dkv_groups.DkvGroups(*found) == expected
    assert list(found[0]) == list(expected.groups)


def test_the_module_is_built():
    assert native._plan_analysis is not None


@pytest.mark.parametrize("name", list(CASES))
def test_plans_of_the_planner(name):
    for plan in _plans(name):
        _same_direct(plan)
        for limit in (2, 3, 8, 32):
            for analysed in (direct.DirectPlan(), direct._analyse_any(plan)):
                _same_groups(plan, limit, analysed)


def _changed(plan, rng):
    """The plan with a few blocks, ops and pairs exchanged, dropped, repeated or of another size or type."""
    plan = copy.copy(plan)
    plan.instructions = instrs = [copy.copy(i) for i in plan.instructions]

    def other(block):
        how = rng.randrange(4)
        if how == 0:
            return BufferBlock(block.buffer_type, max(0, block.index + rng.choice((-1, 1, 40))), block.n_tokens)
        if how == 1:
            return BufferBlock(block.buffer_type, block.index, block.n_tokens + rng.choice((-1, 1)))
        if how == 2:
            return BufferBlock(rng.choice([v for k, v in vars(BufferType).items() if k[:2] in ("LO", "BU")]), block.index, block.n_tokens)
        return BufferBlock(str(b"".join([block.buffer_type.encode()]), "ascii"), block.index, block.n_tokens)  # a string of its own

    def in_list(items, change):
        items = list(items)
        if not items:
            return items
        at, how = rng.randrange(len(items)), rng.randrange(6)
        if how == 0:
            items.insert(rng.randrange(len(items)), items[at])
        elif how == 1 and len(items) > 1:
            del items[at]
        elif how == 2:
            rng.shuffle(items)
        else:
            items[at] = change(items[at])
        return items

    for _ in range(rng.randint(1, 6)):
        instr = rng.choice(instrs)
        if isinstance(instr, MemcpyInstr):
            instr.src_dst_pairs = in_list(instr.src_dst_pairs, lambda p: (other(p[0]), p[1]) if rng.random() < 0.5 else (p[0], other(p[1])))
        elif isinstance(instr, (AttnInstr, AttnBackwardInstr)):
            names = ["q_block_table", "kv_block_table", "out_block_table"]
            names += ["dq_block_table", "dkv_block_table"] if isinstance(instr, AttnBackwardInstr) else []
            name = rng.choice(names)
            table = [list(row) for row in getattr(instr, name)]
            row = table[rng.randrange(len(table))]
            at = rng.randrange(len(row))
            row[at] = other(row[at])
            setattr(instr, name, table)
        elif isinstance(instr, SumInstr):
            instr.ops = in_list(instr.ops, lambda op: SumOp(in_list(op.src_buffers, other), op.dst_buffer) if rng.random() < 0.5
                                else SumOp(op.src_buffers, other(op.dst_buffer)))
        elif isinstance(instr, AttnReductionInstr):
            instr.ops = in_list(instr.ops, lambda op: ReductionOp(in_list(op.src_buffers, lambda p: p), op.dst_buffer))
    if rng.random() < 0.2:
        instrs.insert(rng.randrange(len(instrs) + 1), copy.copy(rng.choice(instrs)))
    return plan


@pytest.mark.parametrize("name", list(CASES))
def test_changed_plans(name):
    rng = random.Random(name)
    taken = 0
    for plan in _plans(name):
        for _ in range(60):
            changed = _changed(plan, rng)
            try:
                expected = direct._analyse_any(changed)
            except (IndexError, TypeError, AttributeError):
                assert native.direct(changed.instructions) is None  # the Python code raises it
                continue
            found = native.direct(changed.instructions)
            if found is not None:
                taken += 1
                assert direct.DirectPlan(*found) == expected
            for limit in (2, 5, 32):
                try:
                    _ = dkv_groups._analyse_any(changed, expected, {i: limit for i, x in enumerate(changed.instructions) if isinstance(x, AttnBackwardInstr)},
                                                {i: (1, 1) for i, x in enumerate(changed.instructions) if isinstance(x, AttnBackwardInstr)}, 1)
                except (IndexError, KeyError):
                    continue
                _same_groups(changed, limit, expected)
    assert taken > 60


def test_what_is_left_to_the_python_code():
    class Block(BufferBlock):
        pass

    class Other:
        ops, output_is_unpadded = [], 0

    block = BufferBlock(BufferType.BUFFER_Q, 3, 128)
    local = BufferBlock(BufferType.LOCAL_Q, 3, 128)
    for bad in (Block(BufferType.BUFFER_Q, 3, 128), BufferBlock("AnotherBuffer", 3, 128), BufferBlock(BufferType.BUFFER_Q, -1, 128),
                BufferBlock(BufferType.BUFFER_Q, 1 << 40, 128), BufferBlock(BufferType.BUFFER_Q, 1 << 70, 128), BufferBlock(BufferType.BUFFER_Q, True, 128)):
        assert native.direct([MemcpyInstr([(local, block)])]) is not None
        assert native.direct([MemcpyInstr([(local, bad)])]) is None
    assert native.direct([MemcpyInstr([(local, block, block)])]) is None
    assert native.direct([MemcpyInstr(iter([(local, block)]))]) is None
    assert native.direct([SumInstr([], 0)]) is not None and native.direct([Other()]) is None
    assert native.direct([BarrierInstr()]) is None
    with pytest.raises(AttributeError):
        instr = MemcpyInstr([(local, block)])
        del instr.src_dst_pairs
        native.direct([instr])


def test_padded_tables():
    rng = random.Random(0)
    cu = [rng.randrange(1 << 30) for _ in range(50)]
    for width in (1, 3, 17):
        rows = [[rng.randrange(50) for _ in range(rng.randint(0, width))] for _ in range(40)]
        blocks = [[BufferBlock(BufferType.BUFFER_KV, i, 1) for i in row] for row in rows]
        for got, expected in ((native.padded(rows, width, cu), executor._padded([[cu[i] for i in row] for row in rows], width)),
                              (native.padded(blocks, width), executor._padded(rows, width))):
            assert got.dtype == np.int32 and np.array_equal(got, expected)
    single = [rng.randrange(50) for _ in range(9)]
    assert np.array_equal(native.padded(single, 1, cu), [[cu[i]] for i in single])
    assert np.array_equal(native.padded(single, 3, cu), [[cu[i], -1, -1] for i in single])
    block = BufferBlock(BufferType.BUFFER_KV, 1 << 31, 1)
    for rows, width, starts in (([[0, 1]], 1, cu), ([[50]], 1, cu), ([[-1]], 1, cu), ([0, [1]], 1, cu), ([[0]], 1, [1 << 31]), ([], 1, cu),
                                ([[]], 0, cu), ([[block]], 1, None), ([[0]], 1, None)):
        assert native.padded(rows, width, starts) is None


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("limit", [2, 32])
def test_the_plan_is_read_before_anything_of_pythons_runs(name, limit):
    """The groups are instances of a class of Python's, whose code may change the plan, or let a thread in that
    does: the plan has been read by then."""
    plan = copy.deepcopy(_plans(name)[1])
    instrs = plan.instructions
    limits = [limit if isinstance(i, AttnBackwardInstr) else 1 for i in instrs]
    analysed = direct._analyse_any(plan)
    expected = native.dkv(copy.deepcopy(instrs), limits, copy.deepcopy(analysed.redirect_ops), dkv_groups.Group)

    class Emptying(dkv_groups.Group):
        __eq__ = dkv_groups.Group.__eq__

        def __init__(self, *args):
            super().__init__(*args)
            for i in instrs:
                if isinstance(i, AttnBackwardInstr):
                    for row in i.kv_block_table + i.dkv_block_table:
                        row[:] = [BufferBlock(BufferType.BUFFER_dKV, 0, 1)]
                elif isinstance(i, SumInstr):
                    for op in i.ops:
                        op.src_buffers, op.dst_buffer = [], None
            for ops in analysed.redirect_ops.values():
                ops.clear()

    fields = lambda groups: {i: [(g.visits, g.dst) for g in of] for i, of in groups.items()}
    found = native.dkv(instrs, limits, analysed.redirect_ops, Emptying)
    assert fields(found[0]) == fields(expected[0]) and found[1:] == expected[1:]
    assert all(not op.src_buffers for i in instrs if isinstance(i, SumInstr) for op in i.ops)  # (it was changed)


def test_a_flag_with_a_truth_of_its_own_is_left_to_the_python_code():
    class Flag:
        def __bool__(self):
            raise AssertionError("asked while the plan is read")

    for flag, taken in ((0, True), (1, True), (True, True), (-3, True), (np.int64(1), False), (None, False), (Flag(), False)):
        assert (native.direct([SumInstr([], flag)]) is not None) == taken
    block, local = BufferBlock(BufferType.BUFFER_dKV, 3, 128), BufferBlock(BufferType.LOCAL_dKV, 3, 128)
    back = AttnBackwardInstr.__new__(AttnBackwardInstr)
    back.kv_block_table, back.dkv_block_table = [[block]], [[block]]
    for flag, taken in ((1, True), (Flag(), False)):
        assert (native.dkv([back, SumInstr([SumOp([block], local)], flag)], [2, 1], {}, dkv_groups.Group) is not None) == taken


def test_high_slot_numbers_cost_no_more_than_in_python():
    """What the native analysis keeps per slot number is kept once, not once a sum op (3200 of the ops here are added in
    part: 0.57 s with a map each, 0.08 with one, in Python 0.11)."""
    plan = make_case(seqlens=[384] * 800, block_size=128, n_heads=4, n_groups=4, head_dim=64, head_block=1)["bw"]
    high = lambda b: BufferBlock(b.buffer_type, b.index + 4100000, b.n_tokens) if b.buffer_type == BufferType.BUFFER_dKV else b
    plan.instructions = [copy.copy(i) for i in plan.instructions]
    for i in plan.instructions:
        if isinstance(i, AttnBackwardInstr):
            i.dkv_block_table = [[high(b) for b in row] for row in i.dkv_block_table]
        elif isinstance(i, SumInstr):
            i.ops = [SumOp([high(b) for b in op.src_buffers], high(op.dst_buffer)) for op in i.ops]
    analysed = direct._analyse_any(plan)
    _same_groups(plan, 2, analysed)
    limits = {i: 2 for i, x in enumerate(plan.instructions) if isinstance(x, AttnBackwardInstr)}

    def seconds(analysis):
        begin = time.process_time()
        analysis()
        return time.process_time() - begin

    by_instr = [limits.get(i, 1) for i in range(len(plan.instructions))]
    natively = min(seconds(lambda: native.dkv(plan.instructions, by_instr, analysed.redirect_ops, dkv_groups.Group)) for _ in range(3))
    in_python = min(seconds(lambda: dkv_groups._analyse_any(plan, analysed, limits, {i: (1, 1) for i in limits}, 1)) for _ in range(3))
    assert natively < 2.5 * in_python, (natively, in_python)
