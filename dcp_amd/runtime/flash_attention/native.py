"""The analyses of a plan in native code (``csrc/python/plan_analysis.cpp``).

Each function answers for the plans that planners make -- instructions, blocks and ops of this package's own
classes, in lists and tuples, with plain integers -- and returns None for any other, which the Python code next
to its caller takes; and None for every plan where the module has not been built."""

from __future__ import annotations

from typing import Optional, Sequence

import numpy as np

from dcp_amd.core import instructions as plans

try:
    from dcp_amd import _plan_analysis
except ImportError:
    _plan_analysis = None
else:
    _plan_analysis.use_types(plans.BufferBlock, plans.ReductionOp, plans.SumOp)

_KINDS = {
    plans.MemcpyInstr: 0,
    plans.CommLaunchInstr: 1,
    plans.BarrierInstr: 2,
    plans.CommWaitInstr: 3,
    plans.AttnInstr: 4,
    plans.AttnBackwardInstr: 5,
    plans.AttnReductionInstr: 6,
    plans.SumInstr: 7,
}


def _kinds(instrs: Sequence) -> Optional[list]:
    if _plan_analysis is None:
        return None
    kinds = [_KINDS.get(type(instr)) for instr in instrs]
    return None if None in kinds else kinds


def direct(instrs: Sequence):
    """The fields of a ``DirectPlan``."""
    kinds = _kinds(instrs)
    return None if kinds is None else _plan_analysis.direct(instrs, kinds)


def dkv(instrs: Sequence, limits: Sequence[int], redirect_ops: dict, group: type):
    """The first three fields of ``DkvGroups``; ``limits``: how many rows a group of an instruction's may visit, ``group``:
    the class of its groups."""
    kinds = _kinds(instrs)
    return None if kinds is None else _plan_analysis.dkv(instrs, kinds, limits, redirect_ops, group)


def padded(rows: Sequence, width: int, cu: Optional[Sequence[int]] = None) -> Optional[np.ndarray]:
    """``rows`` as an int32 table of ``width`` columns, filled up with -1: the slots of rows of blocks or, with ``cu``,
    its values at rows of numbers (at one number a row)."""
    if _plan_analysis is None or not rows or width < 1:
        return None
    table = np.empty((len(rows), width), dtype=np.int32)
    return table if _plan_analysis.padded(rows, width, cu, int(cu is not None and not isinstance(rows[0], list)), table) else None
