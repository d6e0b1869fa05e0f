"""Which copies of a plan the executor need not make.

A plan spells out every block movement: a ``MemcpyInstr`` gathers the device's own blocks from the
unpadded ``LOCAL_*`` tensors into padded ``BUFFER_*`` slots before the attention kernels read them
(reference ``_copy_input_to_local_buffer``, ``dcp/core/scheduler.py:870-892``), and the final
``AttnReductionInstr`` / ``SumInstr`` with ``output_is_unpadded=1`` moves results back
(``scheduler.py:1764-1940``).  Where such a movement is a plain copy -- a slot that holds nothing but
a local block and is read by attention kernels only; a partial output, dQ or summed dK/dV that a
single-source op scatters back unchanged -- the kernels can address the unpadded tensor itself: a
block table entry becomes a token offset (``local_cu_seqlens``) instead of a slot number, the stride
of a table entry a token instead of a block (``dcp_attn_fwd_strided`` / ``dcp_attn_bwd_strided``).
The bytes that reach ``LOCAL_OUT``, ``LOCAL_LSE``, ``LOCAL_dQ`` and ``LOCAL_dKV`` are the same: the
skipped operations are bit copies (and a sum that is rounded once is rounded once either way).

``analyse`` only looks at the instruction list; it changes nothing in the plan.  Plans that exchange
blocks with other devices are left alone (their slots are also read and written by the exchange).
"""

from __future__ import annotations

from collections import defaultdict
from dataclasses import dataclass, field
from typing import Dict, List, Set, Tuple

from dcp_amd.core.instructions import (
    AttnBackwardInstr,
    AttnInstr,
    AttnReductionInstr,
    BarrierInstr,
    BufferBlock,
    BufferType,
    CommLaunchInstr,
    CommWaitInstr,
    ExecutionPlan,
    MemcpyInstr,
    SumInstr,
)
from dcp_amd.runtime.flash_attention import native


@dataclass
class DirectPlan:
    """Per instruction index, what the executor does differently."""

    # MemcpyInstr: positions of the (src, dst) pairs that are not copied
    skip_pairs: Dict[int, Set[int]] = field(default_factory=dict)
    # AttnInstr / AttnBackwardInstr: operand name ("q", "kv", "out", "dq") -> per row, the index (q, out,
    # dq) or the list of indices (kv) of the LOCAL block(s) the kernel addresses instead of slots.
    # "out" of a forward instruction is where it WRITES; of a backward one where it reads out, lse, dout.
    operands: Dict[int, Dict[str, list]] = field(default_factory=dict)
    # AttnReductionInstr / SumInstr: positions of the ops that are not run
    skip_ops: Dict[int, Set[int]] = field(default_factory=dict)
    # SumInstr: op position -> the LOCAL block the sum is written to instead of its slot
    redirect_ops: Dict[int, Dict[int, BufferBlock]] = field(default_factory=dict)

    def anything(self) -> bool:
        return bool(self.skip_pairs or self.operands or self.skip_ops or self.redirect_ops)


_LOCAL_OF = {
    BufferType.BUFFER_Q: BufferType.LOCAL_Q,
    BufferType.BUFFER_KV: BufferType.LOCAL_KV,
    BufferType.BUFFER_OUT: BufferType.LOCAL_OUT,
    BufferType.BUFFER_LSE: BufferType.LOCAL_LSE,
    BufferType.BUFFER_dOUT: BufferType.LOCAL_dOUT,
}


def analyse(plan: ExecutionPlan) -> DirectPlan:
    instrs = plan.instructions
    if any(isinstance(i, (CommLaunchInstr, CommWaitInstr, BarrierInstr)) for i in instrs):
        return DirectPlan()
    found = native.direct(instrs)
    return _analyse_any(plan) if found is None else DirectPlan(*found)


def _analyse_any(plan: ExecutionPlan) -> DirectPlan:
    """Of any plan; ``native.direct`` does the same for those that planners make."""
    result = DirectPlan()
    instrs = plan.instructions

    # A slot that holds a copy of a local block of the matching type: buffer type -> slot -> (memcpy
    # index, pair position, index and tokens of the local block)
    origin: Dict[str, Dict[int, Tuple[int, int, int, int]]] = defaultdict(dict)
    copied: Dict[int, Set[int]] = {}  # memcpy index -> positions of such copies
    # copied pairs with a reader that does not address them through an operand that can go to the source
    blocked: Set[Tuple[int, int]] = set()
    # results that a scatter may take from their slot: buffer type -> slot -> producer; and the readers of each
    produced: Dict[str, Dict[int, tuple]] = defaultdict(dict)
    readers: Dict[tuple, list] = defaultdict(list)

    # (The tables hold a block per (row, kv block) pair: tens of thousands in a long plan, and a plan is
    # executed once or a few times.  So the loops over them look a block up once and build nothing.)
    def local_rows(buffer_type: str, table):
        """Per row the indices of the local blocks behind its blocks, if every one of them is a fresh copy
        of the matching LOCAL_* type; otherwise the copies among them have a reader in their slot."""
        found = origin[buffer_type].get
        rows = []
        for row in table:
            indices = [h[2] for blk in row if (h := found(blk.index)) is not None and h[3] == blk.n_tokens
                       and blk.buffer_type == buffer_type]
            if len(indices) != len(row):
                for r in table:
                    for b in r:
                        read_in_slot(b)
                return None
            rows.append(indices)
        return rows

    def read_in_slot(blk: BufferBlock):
        h = origin[blk.buffer_type].get(blk.index)
        if h is not None:
            blocked.add((h[0], h[1]))

    def with_entries() -> Set[str]:
        """The buffer types that have blocks in the tables; a block of another type needs no look."""
        return {t for table in (origin, produced) for t, blocks in table.items() if blocks}

    def overwritten(buffer_type: str, index: int):
        origin[buffer_type].pop(index, None)
        produced[buffer_type].pop(index, None)

    candidates: Dict[int, Dict[str, list]] = defaultdict(dict)
    for idx, instr in enumerate(instrs):
        if isinstance(instr, MemcpyInstr):
            of_type = {}
            fresh = copied[idx] = set()
            for pos, (src, dst) in enumerate(instr.src_dst_pairs):
                dst_type = dst.buffer_type
                known = of_type.get(dst_type)
                if known is None:
                    known = of_type[dst_type] = _LOCAL_OF.get(dst_type), origin[dst_type], produced[dst_type]
                local_type, copies, results = known
                if results:
                    results.pop(dst.index, None)
                if src.buffer_type == local_type:
                    copies[dst.index] = (idx, pos, src.index, src.n_tokens)
                    fresh.add(pos)
                elif copies:
                    copies.pop(dst.index, None)
        elif isinstance(instr, (AttnInstr, AttnBackwardInstr)):
            q_local = local_rows(BufferType.BUFFER_Q, [row[:1] for row in instr.q_block_table])
            kv_local = local_rows(BufferType.BUFFER_KV, instr.kv_block_table)
            if q_local is not None:
                candidates[idx]["q"] = [r[0] for r in q_local]
            if kv_local is not None:
                candidates[idx]["kv"] = kv_local
            if isinstance(instr, AttnInstr):
                for b, row in enumerate(instr.out_block_table):
                    for t in (BufferType.BUFFER_OUT, BufferType.BUFFER_LSE):
                        overwritten(t, row[0].index)
                    produced[BufferType.BUFFER_OUT][row[0].index] = ("out", idx, b)
            else:
                # out, lse and dout of a row share the slot number: all three must be copies of the same local block
                types = (BufferType.BUFFER_OUT, BufferType.BUFFER_LSE, BufferType.BUFFER_dOUT)
                hits = [[origin[t].get(row[0].index) for row in instr.out_block_table] for t in types]
                tokens = [row[0].n_tokens for row in instr.out_block_table]
                local = [[h[2] for h in per_type] if all(h is not None and h[3] == n for h, n in zip(per_type, tokens)) else None
                         for per_type in hits]
                if local[0] is not None and local[0] == local[1] == local[2]:
                    candidates[idx]["out"] = local[0]
                else:
                    blocked.update((h[0], h[1]) for per_type in hits for h in per_type if h is not None)
                for b, row in enumerate(instr.dq_block_table):
                    overwritten(row[0].buffer_type, row[0].index)
                    produced[row[0].buffer_type][row[0].index] = ("dq", idx, b)
                # (who wrote a dK/dV replica is not asked for: none of them is moved to where it is read)
                known = with_entries()
                if known:
                    for row in instr.dkv_block_table:
                        for blk in row:
                            if blk.buffer_type in known:
                                overwritten(blk.buffer_type, blk.index)
        elif isinstance(instr, AttnReductionInstr):
            for pos, op in enumerate(instr.ops):
                for src_out, src_lse in op.src_buffers:
                    read_in_slot(src_out)
                    read_in_slot(src_lse)
                    who = produced[src_out.buffer_type].get(src_out.index)
                    if who is not None:
                        readers[who].append((idx, pos, len(op.src_buffers), bool(instr.output_is_unpadded)))
                if not instr.output_is_unpadded:
                    for blk in op.dst_buffer:
                        overwritten(blk.buffer_type, blk.index)
                    produced[op.dst_buffer[0].buffer_type][op.dst_buffer[0].index] = ("merged", idx, pos)
        elif isinstance(instr, SumInstr):
            unpadded = bool(instr.output_is_unpadded)
            known = with_entries()
            for pos, op in enumerate(instr.ops):
                for blk in op.src_buffers:
                    if blk.buffer_type in known:
                        who = produced[blk.buffer_type].get(blk.index)
                        if who is not None:
                            readers[who].append((idx, pos, len(op.src_buffers), unpadded))
                        read_in_slot(blk)
                if not unpadded:
                    dst = op.dst_buffer
                    overwritten(dst.buffer_type, dst.index)
                    produced[dst.buffer_type][dst.index] = ("summed", idx, pos)
                    known.add(dst.buffer_type)
        else:  # an instruction this analysis does not know: leave the plan alone
            return DirectPlan()

    def sole_scatter(who):
        """The single-source, unpadded op that is the only reader of a produced block, if that is so."""
        r = readers.get(who, [])
        if len(r) == 1 and r[0][2] == 1 and r[0][3]:
            return r[0][0], r[0][1]
        return None

    for idx, instr in enumerate(instrs):
        if isinstance(instr, AttnInstr):
            hits = [sole_scatter(("out", idx, b)) for b in range(len(instr.out_block_table))]
            if hits and all(h is not None for h in hits):
                dsts = [instrs[j].ops[pos].dst_buffer for j, pos in hits]
                if all(d[0].buffer_type == BufferType.LOCAL_OUT and d[1].buffer_type == BufferType.LOCAL_LSE and
                       d[0].n_tokens == row[0].n_tokens for d, row in zip(dsts, instr.out_block_table)):
                    candidates[idx]["out"] = [d[0].index for d in dsts]
                    for j, pos in hits:
                        result.skip_ops.setdefault(j, set()).add(pos)
        elif isinstance(instr, AttnBackwardInstr):
            hits = [sole_scatter(("dq", idx, b)) for b in range(len(instr.dq_block_table))]
            if hits and all(h is not None for h in hits):
                dsts = [instrs[j].ops[pos].dst_buffer for j, pos in hits]
                if all(d.buffer_type == BufferType.LOCAL_dQ and d.n_tokens == row[0].n_tokens
                       for d, row in zip(dsts, instr.dq_block_table)):
                    candidates[idx]["dq"] = [d.index for d in dsts]
                    for j, pos in hits:
                        result.skip_ops.setdefault(j, set()).add(pos)
        elif isinstance(instr, SumInstr) and not instr.output_is_unpadded:
            # a sum into a slot whose only reader scatters it back unchanged: sum straight to where that goes
            for pos, op in enumerate(instr.ops):
                hit = sole_scatter(("summed", idx, pos))
                if hit is None:
                    continue
                dst = instrs[hit[0]].ops[hit[1]].dst_buffer
                if dst.buffer_type.startswith("Local") and dst.n_tokens == op.dst_buffer.n_tokens:
                    result.redirect_ops.setdefault(idx, {})[pos] = dst
                    result.skip_ops.setdefault(hit[0], set()).add(hit[1])

    result.operands = {idx: ops for idx, ops in candidates.items() if ops}
    for idx, pos in blocked:
        copied[idx].discard(pos)
    result.skip_pairs = {idx: pairs for idx, pairs in copied.items() if pairs}  # (a slot nobody reads is not worth filling either)
    return result
