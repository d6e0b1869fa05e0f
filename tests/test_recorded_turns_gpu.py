"""Passes of several devices' plans that are made again in one library call give what a pass in turns gives: with other
inputs, from another stream, after a device has prepared again, and not where a caller's handler takes part."""

import pytest
import torch

from tests.plan_cases import make_multi_case

pytestmark = pytest.mark.gpu

SIZES = dict(seqlens=[700, 130, 260], block_size=128, n_heads=4, n_groups=2, head_dim=64, head_block=2)
PLANS = {
    "two_devices": dict(n_nodes=1, n_devices_per_node=2),
    "two_nodes_two_stages": dict(n_nodes=2, n_devices_per_node=2, n_stages=2),  # a relay on a side stream
    "three_stages": dict(n_nodes=1, n_devices_per_node=3, n_stages=3),
}


def _executors(case, forward=True):
    from dcp_amd.runtime.flash_attention.executor import get_executor
    from dcp_amd.runtime.flash_attention.fabric import LocalFabric

    fabric = LocalFabric(case["n_nodes"], case["n_devices_per_node"])
    exs = [get_executor(case["head_block"], case["head_dim"], None, fw_exec_plan=f, bw_exec_plan=b, fabric=fabric)
           for f, b in zip(case["fw"], case["bw"])]
    for ex in exs:
        if not forward:
            ex.mode = "Backward"
        ex.prepare(forward=forward)
    return exs


def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    random = lambda info: torch.randn(info.buffer_shape, generator=g, device="cuda").to(torch.bfloat16)
    return [[random(plan.buffer_info[name]) for name in ("LocalQ", "LocalKV", "LocalQ", "LocalQ")] for plan in case["fw"]]


def _give(exs, inputs, forward):
    for ex, (q, kv, out, dout) in zip(exs, inputs):
        ex.init_forward_input(q, kv)
        if not forward:
            ex.set_local_out_lse(out, torch.full_like(ex.buffers["LocalLSE"], 2.0))
            ex.init_backward_input(dout)


def _results(exs, forward):
    names = ("LocalOut", "LocalLSE") if forward else ("LocaldQ", "LocaldKV")
    return [ex.buffers[name].clone() for ex in exs for name in names]


def _same(a, b):
    return all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("forward", [True, False])
@pytest.mark.parametrize("name", list(PLANS))
def test_later_passes(gpu, name, forward):
    from dcp_amd.runtime.flash_attention import fabric as module

    case = make_multi_case(**SIZES, **PLANS[name])
    want = []
    for seed in (1, 2):
        exs = _executors(case, forward)
        _give(exs, _inputs(case, seed), forward)
        module.execute_together(exs, forward)
        want.append(_results(exs, forward))
    assert exs[0].fabric.recorded[forward]._sequence is None  # made when it is asked for
    for turn, seed in enumerate((1, 2, 2, 1)):
        _give(exs, _inputs(case, seed), forward)
        if turn == 2:
            stream = torch.cuda.Stream()
            stream.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(stream):
                module.execute_together(exs, forward)
                got = _results(exs, forward)
            torch.cuda.current_stream().wait_stream(stream)
        else:
            module.execute_together(exs, forward)
            got = _results(exs, forward)
        assert exs[0].fabric.recorded[forward]._sequence is not None
        assert _same(got, want[seed - 1])
    # a device prepares again: its buffers, tables and staging are new ones
    exs[1].prepare(forward=forward)
    before = exs[0].fabric.recorded[forward]
    for _ in range(3):
        _give(exs, _inputs(case, 1), forward)
        module.execute_together(exs, forward)
        assert _same(_results(exs, forward), want[0])
    assert exs[0].fabric.recorded[forward] is not before
    # a synchronous executor goes through its instructions
    waits = []
    exs[0].register_synchronization_handler(lambda: (waits.append(1), torch.cuda.synchronize()))
    exs[0].synchronous = True
    _give(exs, _inputs(case, 2), forward)
    module.execute_together(exs, forward)
    assert len(waits) == len((case["fw"] if forward else case["bw"])[0].instructions)
    assert _same(_results(exs, forward), want[1])


def test_a_handler_of_the_callers_own(gpu):
    from dcp_amd.core.instructions import CommWaitInstr
    from dcp_amd.runtime.flash_attention import executor, fabric as module

    case = make_multi_case(**SIZES, **PLANS["two_devices"])
    exs = _executors(case)
    seen = []
    exs[1]._handlers._by_type[CommWaitInstr] = lambda e, i: (seen.append(i.key), executor._handle_comm_wait(e, i))
    _give(exs, _inputs(case, 1), True)
    for _ in range(3):
        module.execute_together(exs)
    assert len(seen) == 3 * sum(isinstance(i, CommWaitInstr) for i in case["fw"][1].instructions)
    assert not exs[0].fabric.recorded
