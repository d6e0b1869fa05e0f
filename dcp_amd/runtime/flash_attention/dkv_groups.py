"""Which dK/dV replicas of a plan the backward kernel adds up itself.

A plan gives every (attention row, kv block) pair a private dK/dV block and adds the replicas of a
kv block with ``SumInstr`` ops afterwards (reference ``dcp/core/scheduler.py:1365-1700,1764-1940``).
The key-outer kernel holds dK/dV of 128 keys in registers, so rows of one launch that attend to the
same kv block can be visited one after the other by the workgroup that holds its keys
(``dcp_attn_bwd_grouped``): K and V are loaded once, the replicas are added in fp32 without being
rounded and written first, and a sum whose sources have all been added that way is not run.

Where a plan is so small that its (row, kv block) pairs leave most of the device idle, the opposite: a
pair's queries are split over several workgroups (``Group.heads``, ``Group.tiles``), whose shares are
left in fp32 and added, and rounded once, by the sum that would have added the replicas.

``analyse`` looks at the instruction list only and changes nothing in the plan.  It takes replicas
together that one ``SumInstr`` op reads and nothing else does; what that op still has to add are the
groups' first slots and whatever other sources it has (blocks received from other devices, ...).
"""

from __future__ import annotations

import math
from collections import Counter, defaultdict
from dataclasses import dataclass, field
from typing import Dict, List, Optional, Set, Tuple, Union

from dcp_amd.core.instructions import (
    AttnBackwardInstr,
    AttnInstr,
    AttnReductionInstr,
    BarrierInstr,
    BufferBlock,
    BufferType,
    CommLaunchInstr,
    CommType,
    CommWaitInstr,
    ExecutionPlan,
    MemcpyInstr,
    SumInstr,
)
from dcp_amd.runtime.flash_attention import native
from dcp_amd.runtime.flash_attention.direct import DirectPlan

MAX_VISITS = 32  # DCP_ATTN_BWD_MAX_VISITS


@dataclass
class Group:
    """Rows of one launch that attend to one kv block: ``(row, position in the row's kv blocks)``."""

    visits: List[Tuple[int, int]]
    # a BUFFER_dKV slot, or the LOCAL_dKV block the sum would have been scattered to, or the number of a
    # partial (fp32, a block each)
    dst: Union[BufferBlock, int]
    heads: Tuple[int, int] = (0, 0)  # of each kv head's q heads [begin, end); (0, 0): all
    tiles: Tuple[int, int] = (0, 0)  # (n, i): every n-th 64-query tile from the i-th on; (0, 0): all


@dataclass
class DkvGroups:
    # AttnBackwardInstr -> its groups, the ones with the most visits first
    groups: Dict[int, List[Group]] = field(default_factory=dict)
    # SumInstr -> positions of the ops that are not run
    skip_ops: Dict[int, Set[int]] = field(default_factory=dict)
    # SumInstr -> op position -> the sources the op still adds
    sources: Dict[int, Dict[int, List[BufferBlock]]] = field(default_factory=dict)
    # SumInstr -> op position -> the partials the op adds instead
    partials: Dict[int, Dict[int, List[int]]] = field(default_factory=dict)
    n_partials: int = 0


def visits_per_group(n_visits: int, tiles_per_visit: int, n_slots: int) -> int:
    """How many rows a workgroup may visit.  Longer groups save prologues, K/V loads and replicas;
    but a launch is as long as its longest workgroup, and too few of them leave the device idle.  Up
    to eight (row, kv block) pairs per workgroup slot of the device, groups of as many, so that (nearly) all
    of them run at once: rounded up to three, to the nearest past that (at 3.1 pairs three rows beat four by
    5 %; between the points measured the choice is within a few percent either way).  Past eight half
    as many, so that the slots, which take the longest groups first, end within a fraction of a group of
    each other.  Measured, backward (us) with 1 / 2 / 3 / 4 / 6 / 8 rows per group: 1.2 pairs per slot (4096
    tokens, 32 heads) 266 / 249 / 303 / 358 / 357 / 358; 1.9 (4096 tokens, 8 heads of size 64) 95 / 80 / 80 /
    84 / 95 / 101; 2.6 (20000 tokens, 8 heads) 547 / 514 / 509 / 532 / 616 / 716; 3.1 (8192 tokens, 32 heads)
    902 / 848 / 840 / 880 / 975 / 980; 3.5 (16384 tokens, 16 heads) 627 / 576 / 565 / 558 / 639 / 724; 7.1
    (8192 tokens, 8 one-head blocks) 332 / 252 / 237 / 235 / 237 / 232; 7.8 (16384 tokens, 32 heads) 2260 / 2193 /
    2190 / 2161 / 2142 / 2146.  At 25 pairs per slot (32768 tokens, 8 one-head blocks), dK/dV kernel plus
    replica sums 904 in groups of 25 rows and 873 of 13; at 32 (65536 tokens, 32 heads) 8226 and 8330."""
    pairs = n_visits * tiles_per_visit / n_slots
    if pairs <= 8:
        return max(1, math.ceil(pairs) if pairs <= 3 else round(pairs))
    return min(MAX_VISITS, max(8, math.ceil(pairs / 2)))


def parts_per_visit(n_visits: int, tiles_per_visit: int, n_slots: int, n_heads: int, n_q_tiles: int) -> Tuple[int, int]:
    """Into how many parts the queries of a (row, kv block) pair are split, by heads and by 64-query
    tiles, so that the launch comes to one workgroup per slot of the device; parts of fewer than four
    steps are not worth their start."""
    steps = n_heads * n_q_tiles
    parts = min(n_slots // max(1, n_visits * tiles_per_visit), steps // 4)
    by_heads = max(1, min(parts, n_heads))
    return by_heads, max(1, min(parts // by_heads, n_q_tiles))


def _visit_order(counts: List[int]):
    """In which order a group visits its rows, as a sort key over row numbers.  Workgroups that run at
    the same time should read the same Q and dO.  With a causal mask every kv block of a sequence is
    seen by its last row: last row first (against first row first 8.29 to 8.50 ms for the dK/dV
    kernel on 65536 causal tokens).  With a sliding window most kv blocks are seen by the same number
    of rows, each by the next ones in turn; taken modulo that number, neighbouring blocks visit a row
    at the same time (131072 tokens, window 4096: 16.6 against 17.1 ms)."""
    number, times = Counter(counts).most_common(1)[0]
    if number > 2 and 2 * times > len(counts):
        return lambda visit: (visit[0] % number, -visit[0])
    return lambda visit: -visit[0]


def _chunk_sizes(n_visits: int, limit: int) -> List[int]:
    """How a kv block with more rows than a group may visit is split: whole groups, then what is left in
    halves down to an eighth of one.  Groups of one size end together and leave the device idle for up
    to a group's time; small ones, handed out last, fill that (98304 tokens, shared prefixes, up to 150
    rows a block: dK/dV kernel and sums 28.2 ms in equal parts of up to 32, 27.5 this way)."""
    sizes = [limit] * (n_visits // limit - 1)
    left = n_visits - sum(sizes)  # between one and two groups
    smallest = max(1, limit // 8)
    while left > 0:
        size = min(limit, max(smallest, (left + 1) // 2))
        sizes.append(min(size, left))
        left -= sizes[-1]
    return sizes


def _components(kv_rows: List[List[int]]) -> Dict[int, Tuple[int, int]]:
    """kv block -> (component, rank in it), two blocks being in one component if some row attends to
    both: the blocks of a sequence's kv head.  In order of first appearance."""
    parent: Dict[int, int] = {}

    def root(x):
        while parent[x] != x:
            parent[x] = x = parent[parent[x]]
        return x

    known = parent.get
    for blocks in kv_rows:
        if not blocks:  # a row that attends to nothing
            continue
        first = blocks[0]
        if first not in parent:
            parent[first] = first
        r = root(first)
        for i in blocks:
            up = known(i)
            if up is None:
                parent[i] = r
            elif up != r and root(i) != r:
                parent[root(i)] = r
    numbers: Dict[int, int] = {}
    ranks: Counter = Counter()
    found = {}
    for i in parent:
        r = root(i)
        found[i] = (numbers.setdefault(r, len(numbers)), ranks[r])
        ranks[r] += 1
    return found


class _Visits:
    """Every (row, kv block) pair of the plan's backward instructions, numbered.  (Tens of thousands in a
    long plan, and a plan is executed once or a few times: the analysis works on these numbers and on
    flat lists, and looks at a block once.)"""

    def __init__(self, instrs):
        self.begin: Dict[int, int] = {}  # instruction -> its first visit
        self.row: List[int] = []
        self.pos: List[int] = []
        self.slot: List[BufferBlock] = []  # the pair's dK/dV replica
        for idx, instr in enumerate(instrs):
            if isinstance(instr, AttnBackwardInstr):
                self.begin[idx] = len(self.row)
                for row, blocks in enumerate(instr.dkv_block_table):
                    self.row += [row] * len(blocks)
                    self.pos += range(len(blocks))
                    self.slot += blocks

    def of(self, idx: int, instr: AttnBackwardInstr) -> range:
        return range(self.begin[idx], self.begin[idx] + sum(map(len, instr.dkv_block_table)))


_UNREAD, _ELSEWHERE = -1, -2  # readers of a replica: none; other than one sum op

# the instructions whose reads and writes of BUFFER_dKV slots `analyse` follows
_KNOWN = {AttnInstr, AttnBackwardInstr, AttnReductionInstr, BarrierInstr, CommLaunchInstr, CommWaitInstr, MemcpyInstr, SumInstr}


def analyse(plan: ExecutionPlan, direct: DirectPlan, n_heads_kv: int, tiles_per_block: int, n_slots: int,
            q_heads_per_kv_head: int = 1) -> DkvGroups:
    result = DkvGroups()
    instrs = plan.instructions
    if not _KNOWN.issuperset(map(type, instrs)):  # an instruction of another kind may read any replica
        return result
    limits, parts = {}, {}
    for idx, instr in enumerate(instrs):
        if isinstance(instr, AttnBackwardInstr):
            n_visits = sum(map(len, instr.dkv_block_table))
            limits[idx] = visits_per_group(n_visits, tiles_per_block * n_heads_kv, n_slots)
            parts[idx] = (1, 1) if limits[idx] > 1 else parts_per_visit(
                n_visits, tiles_per_block * n_heads_kv, n_slots, q_heads_per_kv_head, 2 * tiles_per_block)
    if all(limit == 1 for limit in limits.values()) and all(p == (1, 1) for p in parts.values()):
        return result
    if all(p == (1, 1) for p in parts.values()):  # (launches in parts have few pairs)
        found = native.dkv(instrs, [limits.get(idx, 1) for idx in range(len(instrs))], direct.redirect_ops, Group)
        if found is not None:
            return DkvGroups(*found)
    return _analyse_any(plan, direct, limits, parts, q_heads_per_kv_head)


def _analyse_any(plan: ExecutionPlan, direct: DirectPlan, limits: Dict[int, int], parts: Dict[int, Tuple[int, int]],
                 q_heads_per_kv_head: int) -> DkvGroups:
    """Of any plan; ``native.dkv`` does the same for those that planners make, where no launch is in parts."""
    result = DkvGroups()
    instrs = plan.instructions
    visits = _Visits(instrs)
    row_of, pos_of, slot_of = visits.row, visits.pos, visits.slot
    # which visit wrote a BUFFER_dKV slot last, if a backward kernel did, and which sum op reads what it wrote
    written: Dict[int, int] = {}
    reader = [_UNREAD] * len(row_of)
    sum_ops: List[Tuple[int, int]] = []  # the sum ops, numbered as in `reader`: (instruction, position)
    replicas_of: Dict[int, List[int]] = defaultdict(list)  # what a sum op reads of that kind
    dkv, local_dkv = followed = (BufferType.BUFFER_dKV, BufferType.LOCAL_dKV)
    named: Counter = Counter()  # how often the plan names a LOCAL_dKV block
    in_parts = {idx for idx, p in parts.items() if p != (1, 1)}

    def reads(blocks, who=_ELSEWHERE):
        for block in blocks:
            if block.buffer_type == dkv:
                replica = written.get(block.index)
                if replica is not None:
                    reader[replica] = who if reader[replica] == _UNREAD else _ELSEWHERE
                    if in_parts:
                        replicas_of[who].append(replica)
            elif block.buffer_type == local_dkv:
                named[block.index] += 1

    def writes(block: BufferBlock):
        if block.buffer_type == dkv:
            written.pop(block.index, None)
        elif block.buffer_type == local_dkv:
            named[block.index] += 1

    for idx, instr in enumerate(instrs):
        if isinstance(instr, AttnBackwardInstr):
            mine = visits.of(idx, instr)
            written.update(zip([block.index for block in slot_of[mine.start : mine.stop]], mine))
        elif isinstance(instr, SumInstr):
            for pos, op in enumerate(instr.ops):
                reads(op.src_buffers, len(sum_ops))
                sum_ops.append((idx, pos))
            for op in instr.ops:
                writes(op.dst_buffer)
        elif isinstance(instr, MemcpyInstr):
            for src, dst in instr.src_dst_pairs:
                if src.buffer_type in followed or dst.buffer_type in followed:
                    reads((src,))
                    writes(dst)
        elif isinstance(instr, CommLaunchInstr):
            for op in instr.comm_ops:
                # (a receive lands at the wait at the latest: the slot is the exchange's from here on)
                if op.comm_type == CommType.SEND:
                    reads((op.buffer_block,))
                else:
                    writes(op.buffer_block)
        elif isinstance(instr, AttnReductionInstr):
            for op in instr.ops:
                for blocks in op.src_buffers:
                    reads(blocks)
                for block in op.dst_buffer:
                    writes(block)

    # sum ops all of whose sources can be left as partials
    splittable = {v for idx in in_parts for v in visits.of(idx, instrs[idx])}
    split_ops = {who for who, replicas in replicas_of.items() if who >= 0
                 and len(replicas) == len(instrs[sum_ops[who][0]].ops[sum_ops[who][1]].src_buffers)
                 and all(v in splittable and reader[v] == who for v in replicas)}
    for idx in sorted(in_parts):
        by_heads, by_tiles = parts[idx]
        groups = []
        for v in visits.of(idx, instrs[idx]):
            who, pair = reader[v], (row_of[v], pos_of[v])
            if who not in split_ops:
                groups.append(Group([pair], slot_of[v]))
                continue
            j, op_pos = sum_ops[who]
            for i in range(by_heads):
                heads = (q_heads_per_kv_head * i // by_heads, q_heads_per_kv_head * (i + 1) // by_heads)
                for k in range(by_tiles):
                    groups.append(Group([pair], result.n_partials, heads, (by_tiles, k) if by_tiles > 1 else (0, 0)))
                    result.partials.setdefault(j, {}).setdefault(op_pos, []).append(result.n_partials)
                    result.n_partials += 1
        result.groups[idx] = groups

    for idx, instr in enumerate(instrs):
        if limits.get(idx, 1) == 1:  # the launch does without groups
            continue
        mine = visits.of(idx, instr)
        kv_rows = [[block.index for block in row] for row in instr.kv_block_table]
        kv_of = [i for row in kv_rows for i in row]
        # rows to take together: the same kv block, added by the same op and read by nothing else
        alone: List[int] = []
        together: Dict[Tuple[int, int, int], List[int]] = defaultdict(list)
        for v, kv_block in zip(mine, kv_of):
            if reader[v] < 0:
                alone.append(v)
            else:
                together[reader[v], kv_block, slot_of[v].n_tokens].append(v)
        limit = limits[idx]
        groups: List[Group] = [Group([(row_of[v], pos_of[v])], slot_of[v]) for v in alone]
        if together or alone:
            order = _visit_order([len(t) for t in together.values()] + [1] * len(alone))
        for (who, _, _), taken in together.items():
            taken.sort(key=lambda v: order((row_of[v], pos_of[v])))
            j, op_pos = sum_ops[who]
            op = instrs[j].ops[op_pos]
            dst = direct.redirect_ops.get(j, {}).get(op_pos, op.dst_buffer if instrs[j].output_is_unpadded else None)
            if (len(taken) <= limit and len(taken) == len(op.src_buffers) and dst is not None
                    and dst.buffer_type == local_dkv and dst.n_tokens == slot_of[taken[0]].n_tokens
                    and named[dst.index] == 1):  # (the launch writes it earlier than the sum would)
                groups.append(Group([(row_of[v], pos_of[v]) for v in taken], dst))
                result.skip_ops.setdefault(j, set()).add(op_pos)
                continue
            gone, at = set(), 0
            for size in _chunk_sizes(len(taken), limit) if len(taken) > limit else [len(taken)]:
                chunk = taken[at : at + size]
                at += size
                groups.append(Group([(row_of[v], pos_of[v]) for v in chunk], slot_of[chunk[0]]))
                gone.update([slot_of[v].index for v in chunk[1:]])
            ops = result.sources.setdefault(j, {})
            ops[op_pos] = [b for b in ops.get(op_pos, op.src_buffers) if b.buffer_type != dkv or b.index not in gone]
        # longest first; among equals the same block of every sequence and head together: consecutive
        # groups go to the XCDs in turn, so that the blocks of one head, whose rows are the same, meet on
        # one XCD at about the same time (131072 tokens, window 4096, 8 kv heads: 15.6 -> 15.3 ms)
        component = _components(kv_rows)

        def place(group: Group):
            row, pos = group.visits[0]
            number, rank = component[kv_rows[row][pos]]
            return (-len(group.visits), rank, number)

        groups.sort(key=place)
        result.groups[idx] = groups
    return result
