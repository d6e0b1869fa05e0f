"""Block exchange between the executors of several devices that share one GPU and one process.

The reference moves blocks between devices in three passes per direction: a fused copy packs the
blocks to send into one buffer per dtype, ``dist.all_to_all_single`` moves the buffers, and a
second fused copy unpacks what arrived (``dcp/runtime/flash_attention/executor.py:1583-2074``).
Here the sender's one copy kernel writes its blocks straight into the *receiver's* staging
buffer (on MI355X peers map each other's memory over xGMI; in this build every "device" is an
executor on the same GPU, so the peer's buffer is simply another allocation) and signals with a
stream event; the receiver waits for the events of the peers it expects and unpacks.  Two
passes instead of three, and no collective call.  The staging buffer keeps the reference's
rule that received blocks reach their slots at the ``CommWaitInstr``, not earlier, so slot reuse
planned by the scheduler stays valid.

``LocalFabric`` is the registry the executors meet in: staging buffers by (receiver, key,
dtype), "posted" events by (sender, receiver, key) and "consumed" events by (receiver, key) that
keep a sender of the next iteration from overwriting a staging buffer still being unpacked.
``execute_together`` runs the plans of all devices in turns on the one GPU.
"""

from __future__ import annotations

import weakref
from typing import Dict, List, Optional, Sequence, Tuple

import torch

from dcp_amd import _lib
from dcp_amd.core.instructions import BarrierInstr, CommWaitInstr


class LocalFabric:
    def __init__(self, n_nodes: int, n_devices_per_node: int):
        self.n_nodes = n_nodes
        self.n_devices_per_node = n_devices_per_node
        self.n_ranks = n_nodes * n_devices_per_node
        # (receiver, key, dtype) -> (staging tensor, {sender: (element offset, [block numels])})
        self._staging: Dict[Tuple[int, str, torch.dtype], Tuple[torch.Tensor, Dict[int, Tuple[int, List[int]]]]] = {}
        self._posted: Dict[Tuple[int, int, str], torch.cuda.Event] = {}
        self._consumed: Dict[Tuple[int, str], torch.cuda.Event] = {}
        self._barrier_arrivals = [0] * self.n_ranks
        self.epoch = 0  # changes whenever a staging buffer is (re)registered or dropped
        self.recorded = {}  # forward or not -> RecordedTurns

    # -- prepare time ----------------------------------------------------------------------
    def register_staging(self, receiver: int, key: str, dtype: torch.dtype, staging: torch.Tensor,
                         segments: Dict[int, Tuple[int, List[int]]]) -> None:
        self._staging[(receiver, key, dtype)] = (staging, segments)
        self.epoch += 1

    def staging_segment(self, receiver: int, key: str, dtype: torch.dtype, sender: int):
        """``(staging tensor, element offset, block numels)`` of what ``receiver`` expects from
        ``sender`` under ``key``; raises if the receiver's plan has no such receives."""
        entry = self._staging.get((receiver, key, dtype))
        if entry is None or sender not in entry[1]:
            raise RuntimeError(
                f"rank {sender} sends {dtype} blocks to rank {receiver} under key {key!r}, but rank "
                f"{receiver} has prepared no matching receives (prepare every device before executing)"
            )
        offset, numels = entry[1][sender]
        return entry[0], offset, numels

    def forget(self, receiver: int) -> None:
        """Drop what ``receiver`` registered (its plan is being prepared again)."""
        for k in [k for k in self._staging if k[0] == receiver]:
            del self._staging[k]
        self.epoch += 1

    # -- execute time ----------------------------------------------------------------------
    def post(self, sender: int, receiver: int, key: str, event: torch.cuda.Event) -> None:
        self._posted[(sender, receiver, key)] = event

    def posted(self, sender: int, receiver: int, key: str) -> Optional[torch.cuda.Event]:
        return self._posted.get((sender, receiver, key))

    def take(self, sender: int, receiver: int, key: str) -> torch.cuda.Event:
        return self._posted.pop((sender, receiver, key))

    def consumed(self, receiver: int, key: str) -> Optional[torch.cuda.Event]:
        return self._consumed.get((receiver, key))

    def set_consumed(self, receiver: int, key: str, event: torch.cuda.Event) -> None:
        self._consumed[(receiver, key)] = event

    def barrier_arrive(self, rank: int) -> int:
        self._barrier_arrivals[rank] += 1
        return self._barrier_arrivals[rank]

    def barrier_passed(self, generation: int) -> bool:
        return min(self._barrier_arrivals) >= generation


# what a pass in turns calls on the fabric
_PASS_METHODS = {name: vars(LocalFabric)[name] for name in ("post", "posted", "take", "consumed", "set_consumed")}


def methods_are(obj, methods) -> bool:
    """Are these (name -> function) still what the object calls by these names, whatever a subclass or a caller did?"""
    return all(getattr(getattr(obj, name), "__func__", None) is function for name, function in methods.items())


class RecordedTurns:
    """What ``execute_together`` does in a pass, done again in one library call: the recorded calls of the devices'
    instructions on their streams and the events by which they wait for each other, in the order in which the
    turns of the first pass took them.  Forward and backward of 16384 tokens, 8 heads, four devices: to walk the
    plans' 112 instructions in Python took 2.2 ms a pass, longer than their 150 kernels; the pass took 2130 us
    and takes 1760, which are the kernels'.  That is from the third pass on: the first goes in turns (and packs the
    tables of what is sent), and the second also puts the sequence together, 0.15 ms more than in turns.
    Holds nothing of the executors; ``fits`` says whether all is still as it was.  The events are its own: a pass in
    turns makes new ones."""

    def __init__(self, executors, turns: List[Tuple[int, int]]):
        self._executors = [weakref.ref(ex) for ex in executors]
        self._tokens = [ex.steps_token() for ex in executors]
        self._epoch = executors[0].fabric.epoch
        self._turns = turns
        self._sequence = None  # (made when the second pass asks for it)
        self._events: List[torch.cuda.Event] = []
        self._consumed: Dict[Tuple[int, str], torch.cuda.Event] = {}

    @staticmethod
    def of(executors, plans, turns) -> Optional["RecordedTurns"]:
        """None where some instruction does more than the library's calls, or where an executor or the fabric has methods of
        the caller's own: a pass in turns calls them."""
        if not methods_are(executors[0].fabric, _PASS_METHODS):
            return None
        if not all(hasattr(ex, "turns_are_recordable") and ex.turns_are_recordable(plan) for ex, plan in zip(executors, plans)):
            return None
        return RecordedTurns(executors, turns)

    def fits(self, executors, plans) -> bool:
        return (len(executors) == len(self._executors)
                and all(ref() is ex for ref, ex in zip(self._executors, executors))
                and self._epoch == executors[0].fabric.epoch and methods_are(executors[0].fabric, _PASS_METHODS)
                # (the plans are those of the first pass where the token is the same and the steps are the plan's)
                and all(ex.steps_token() == token and ex.turns_are_recordable(plan)
                        for ex, plan, token in zip(executors, plans, self._tokens))
                and (self._sequence is not None or self._make(executors, plans)))

    def _event(self, stream) -> torch.cuda.Event:
        event = torch.cuda.Event()
        event.record(stream)  # (it exists from here on)
        self._events.append(event)
        return event

    def _make(self, executors, plans) -> bool:
        RUN, RECORD, WAIT = _lib.Sequence.RUN, _lib.Sequence.RECORD, _lib.Sequence.WAIT
        steps = [(rank, executors[rank].recorded_step(plans[rank], i)) for rank, i in self._turns]
        launches = [(rank, step["key"]) for rank, step in steps if step and step["kind"] == "launch"]
        received = {(rank, step["key"]) for rank, step in steps if step and step["kind"] == "wait" and step["peers"]}
        if (any(step is None for _, step in steps) or len(set(launches)) < len(launches)
                or any((peer, step["key"]) not in received for _, step in steps if step["kind"] == "launch" for peer in step["peers"])):
            return False  # a call that is not known, two exchanges of one name, or sends that nobody waits for
        launched: Dict[Tuple[int, str], torch.cuda.Event] = {}
        self._consumed = {(rank, step["key"]): self._event(step["stream"]) for rank, step in steps
                          if step["kind"] == "wait" and step["peers"]}
        begins = self._event(torch.cuda.current_stream())
        ops = [(RECORD, begins, None)] + [(WAIT, begins, ex.main_stream) for ex in executors]
        for rank, step in steps:
            kind, stream, key = step["kind"], step["stream"], step.get("key")
            if kind == "launch":
                if stream != executors[rank].main_stream:  # the blocks to send are produced there
                    ops += self._join(executors[rank].main_stream, stream)
                ops += [(WAIT, self._consumed[peer, key], stream) for peer in step["peers"]]
            elif kind == "wait":
                ops += [(WAIT, launched[peer, key], stream) for peer in [rank] + step["peers"]]
            ops += [(RUN, recording, stream) for recording in step["calls"]]
            if kind == "launch":
                launched[rank, key] = self._event(stream)
                ops.append((RECORD, launched[rank, key], stream))
            elif kind == "wait" and step["peers"]:
                ops.append((RECORD, self._consumed[rank, key], stream))
        for ex in executors:
            for side in ex.streams.values():
                ops += self._join(side, ex.main_stream)
            ops += self._join(ex.main_stream, None)
        self._sequence = _lib.Sequence(ops)
        return True

    def _join(self, stream, follower):
        event = self._event(stream)
        return [(_lib.Sequence.RECORD, event, stream), (_lib.Sequence.WAIT, event, follower)]

    def run(self, executors, plans) -> None:
        caller, fabric = torch.cuda.current_stream(), executors[0].fabric
        for ex, plan in zip(executors, plans):
            ex.begin_recorded(plan, caller)
        for (rank, key), event in self._consumed.items():
            last = fabric.consumed(rank, key)
            if last is not event:  # another kind of pass came before: everybody waits for its unpacking
                if last is not None:
                    for ex in executors:
                        ex.main_stream.wait_event(last)
                fabric.set_consumed(rank, key, event)
        self._sequence.run(caller.cuda_stream)
        for ex in executors:
            ex.finish_recorded(caller)


def execute_together(executors: Sequence, forward: bool = True) -> None:
    """Run the current mode's plan of every executor (``executors[rank]``, all on one
    ``LocalFabric``) to its end.  Each device runs until it reaches a wait whose peers have not
    launched yet (or a barrier not everybody has reached), then the next device takes over; the
    kernels of different devices overlap on the GPU as far as their streams allow."""
    plans = [ex.fw_exec_plan if forward else ex.bw_exec_plan for ex in executors]
    fabric = getattr(executors[0], "fabric", None) if executors else None
    recorded = fabric.recorded.pop(forward, None) if isinstance(fabric, LocalFabric) else None
    if recorded is not None and recorded.fits(executors, plans):
        fabric.recorded[forward] = recorded
        return recorded.run(executors, plans)
    turns: List[Tuple[int, int]] = []  # (rank, instruction) in the order they are taken
    for ex, plan in zip(executors, plans):
        ex.begin(plan)
    cursor = [0] * len(executors)
    while any(c < len(p.instructions) for c, p in zip(cursor, plans)):
        progressed = False
        for rank, (ex, plan) in enumerate(zip(executors, plans)):
            while cursor[rank] < len(plan.instructions):
                instr = plan.instructions[cursor[rank]]
                if isinstance(instr, CommWaitInstr) and not ex.comm_ready(instr.key):
                    break
                if isinstance(instr, BarrierInstr) and not ex.barrier_ready(cursor[rank]):
                    break
                ex.step(cursor[rank])
                turns.append((rank, cursor[rank]))
                cursor[rank] += 1
                progressed = True
        if not progressed:
            raise RuntimeError("the devices' plans wait for each other: no instruction can run")
    for ex in executors:
        ex.finish()
    if isinstance(fabric, LocalFabric):
        recorded = RecordedTurns.of(executors, plans, turns)
        if recorded is not None:
            fabric.recorded[forward] = recorded
