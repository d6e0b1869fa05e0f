"""Later passes of several devices' plans in one library call (``fabric.RecordedTurns``), on the host alone: which passes
may be made that way, and what the sequence is made from.  Two devices, one sends the other a block."""

from contextlib import nullcontext
from types import SimpleNamespace

import pytest
import torch

from dcp_amd.core.executor import HandlerTable
from dcp_amd.core.instructions import CommLaunchInstr, CommWaitInstr, MemcpyInstr
from dcp_amd.runtime.flash_attention import executor as module, fabric


class _Stream:
    device_index, cuda_stream = 0, 1

    def wait_stream(self, other):
        pass

    wait_event = wait_stream


class _Event:
    def record(self, stream):
        pass


class _Sequence:
    RUN, RECORD, WAIT = range(3)
    made, runs = [], 0

    def __init__(self, ops):
        _Sequence.made.append([(kind, what) for kind, what, _ in ops if kind == self.RUN])

    def run(self, stream):
        _Sequence.runs += 1


def _no_launches():
    return module._Copies({}, None)


@pytest.fixture
def devices(monkeypatch):
    """Two executors and their plans: a gather, then one block from the first device to the second."""
    callers = _Stream()
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: callers)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "stream", lambda stream: nullcontext())
    monkeypatch.setattr(torch.cuda, "Event", _Event)
    for name in ("range_push", "range_pop"):
        monkeypatch.setattr(torch.cuda.nvtx, name, lambda *a: None)
    monkeypatch.setattr(fabric._lib, "Sequence", _Sequence)
    _Sequence.made, _Sequence.runs = [], 0
    between = fabric.LocalFabric(1, 2)
    executors = []
    for rank in range(2):
        ex = module.AttentionExecutor.__new__(module.AttentionExecutor)
        ex.node_id, ex.local_device_id, ex.n_devices_per_node, ex.fabric = 0, rank, 2, between
        ex.main_stream, ex.streams, ex.head_dim, ex.kernel_head_dim = _Stream(), {}, 64, 64
        ex.synchronous, ex.logger, ex.buffers, ex.pending_comm_ops = False, None, {}, {}
        ex._last_stream = ex._last_pass = ex._dkv_partials = ex._bwd_workspace = ex._fwd_partials = None
        ex._recorded_steps, ex._steps_of, ex._steps_token = {}, (None, ()), object()
        ex._handlers = HandlerTable("Instruction handler")
        for kind in (MemcpyInstr, CommLaunchInstr, CommWaitInstr):
            ex.register_handler(kind, module._TURN_HANDLERS[kind])
        ex.fw_exec_plan = SimpleNamespace(instructions=[MemcpyInstr([]), CommLaunchInstr("key", []), CommWaitInstr("key")], buffer_info={})
        ex._args_cache = {0: dict(other={}, lse={}), 1: dict(sends=[], pack=_no_launches(), epoch=between.epoch, send_peers=[1] if rank == 0 else [],
                                                 recv_peers=[0] if rank else [], unpack=_no_launches(), staging=[])}
        executors.append(ex)
    return executors


def _counted(calls, inner):
    def counted(*args):
        calls.append(args)
        return inner(*args)

    return counted


def test_passes_after_the_first_are_one_call(devices):
    """(Of plans of any type: these cannot be weakly referenced.)"""
    for turn in range(3):
        fabric.execute_together(devices)
        assert _Sequence.runs == turn


@pytest.mark.parametrize("passes_before", [0, 2])
@pytest.mark.parametrize("how", ["instance", "subclass", "class"])
@pytest.mark.parametrize("name", ["begin", "step", "finish", "comm_ready", "post", "posted", "take", "consumed", "set_consumed"])
def test_methods_of_the_callers_own_run_in_every_pass(devices, monkeypatch, name, how, passes_before):
    """A pass in turns calls them, so a caller may put something of their own in their place, at the start or later."""
    for _ in range(passes_before):
        fabric.execute_together(devices)
    targets, calls = [devices[0].fabric] if hasattr(fabric.LocalFabric, name) else devices, []
    kind = type(targets[0])
    if how == "instance":
        for target in targets:
            setattr(target, name, _counted(calls, getattr(target, name)))
    elif how == "subclass":
        own = type("Own", (kind,), {name: _counted(calls, getattr(kind, name))})
        for target in targets:
            target.__class__ = own
    else:
        monkeypatch.setattr(kind, name, _counted(calls, getattr(kind, name)))
    _Sequence.runs = 0
    fabric.execute_together(devices)
    in_a_pass = len(calls)
    assert in_a_pass > 0
    for _ in range(2):
        fabric.execute_together(devices)
    assert len(calls) == 3 * in_a_pass and _Sequence.runs == 0


def test_a_pass_of_another_plan_between_the_first_and_the_second(devices):
    """The calls are those of the plan that the devices run together, whatever a device ran by itself last."""
    fabric.execute_together(devices)
    for ex in devices:
        ex.cuda_graph, ex._recorded, ex.return_values = None, None, {}
        with pytest.raises(KeyError, match="LocalOut"):  # (what a pass returns: these executors have no buffers)
            ex.execute(SimpleNamespace(instructions=[], buffer_info={}))
    fabric.execute_together(devices)
    assert _Sequence.runs == 1
    assert [what for _, what in _Sequence.made[0]] == [ex._recorded_steps[0][0] for ex in devices]  # the two gathers
