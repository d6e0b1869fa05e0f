"""Recorded library calls (``dcp_record_*``) and the executor's use of them."""

import pytest
import torch

from tests.plan_cases import make_case


def test_recording_is_per_thread_and_bounded():
    """No GPU needed: an empty problem's call returns before it launches anything."""
    from dcp_amd import _lib

    lib = _lib.load()
    rec = _lib.Recording()
    assert rec.begin()
    assert not _lib.Recording().begin()  # this thread records already
    for _ in range(2):
        _lib.call("dcp_fused_copy_varlen", 0, 0, 0, 0, 0, 0, 0, 0, 16, 2, 0)
    rec.end()
    with pytest.raises(AssertionError, match="not recording"):
        rec_again = _lib.Recording()
        _lib.call("dcp_record_end")
        del rec_again
    _lib.call("dcp_fused_copy_varlen", 0, 0, 0, 0, 0, 0, 0, 0, 16, 2, 0)
    assert rec.size() == 2
    rec.run(0, 2, 0)
    with pytest.raises(AssertionError, match="calls 0 to 3 of 2"):
        rec.run(0, 3, 0)
    assert lib.dcp_record_size(None) == 0


def test_a_nested_call_is_recorded_once_and_errors_come_back():
    from dcp_amd import _lib

    rec = _lib.Recording()
    assert rec.begin()
    try:
        with pytest.raises(ValueError, match="head_dim"):  # dcp_attn_fwd calls dcp_attn_fwd_strided
            _lib.call("dcp_attn_fwd", *([0] * 8), 1, 0, 0, 0, 0, 1, 1, 64, 64, 1, 1, 96, 0, 0, 1, 1.0, 0, 0, 0, 0)
    finally:
        rec.end()
    assert rec.size() == 1
    with pytest.raises(ValueError, match="head_dim"):
        rec.run(0, 1, 0)


def _executors(case):
    from dcp_amd.runtime.flash_attention.executor import get_executor

    ex = get_executor(case["head_block"], case["head_dim"], None, fw_exec_plan=case["fw"], bw_exec_plan=case["bw"])
    ex.prepare(forward=True)
    return ex


CASE = dict(seqlens=[700, 130], block_size=128, n_heads=4, n_groups=2, head_dim=128, head_block=2, n_kv_groups=2, qkv_scale=0.5)


@pytest.mark.gpu
def test_passes_after_the_first_see_new_inputs_and_replaced_buffers(gpu):
    case = make_case(**CASE)
    other = make_case(**CASE, seed=3)
    ex, fresh = _executors(case), _executors(case)
    inputs = [(c["layout"].to_local_q(c["q"]).cuda(), c["layout"].to_local_kv(c["kv"]).cuda()) for c in (case, other)]
    first = ex.forward(*inputs[0])
    assert ex._recorded is not None
    second = ex.forward(*inputs[1])  # the recorded calls, other inputs
    want = fresh.forward(*inputs[1])
    again = ex.forward(*inputs[0])
    assert all(torch.equal(a, b) for a, b in zip(second, want))
    assert all(torch.equal(a, b) for a, b in zip(first, again))
    # a buffer the caller replaced: the kernels that read it through the executor see the new one
    ex.buffers["LocalLSE"] = torch.full_like(ex.buffers["LocalLSE"], 7.0)
    replaced = ex.forward(*inputs[1])
    assert all(torch.equal(a, b) for a, b in zip(replaced, want))


@pytest.mark.gpu
def test_passes_on_another_stream_wait_for_the_last_one(gpu):
    case = make_case(**CASE)
    ex = _executors(case)
    q, kv = case["layout"].to_local_q(case["q"]).cuda(), case["layout"].to_local_kv(case["kv"]).cuda()
    want = ex.forward(q, kv)
    torch.cuda.synchronize()
    ex.buffers["LocalOut"].zero_()
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    with torch.cuda.stream(streams[0]):
        torch.cuda._sleep(20_000_000)
        ex.execute(case["fw"], True)
        marker = torch.cuda.Event()
        marker.record()
    with torch.cuda.stream(streams[1]):
        ex.buffers["LocalLSE"]  # (no work of its own on this stream)
        out, lse = ex.execute(case["fw"], True)
        out, lse = out.clone(), lse.clone()
        done = torch.cuda.Event()
        done.record()
    done.synchronize()
    assert marker.query()  # the pass on the first stream was over before the second one ran
    assert torch.equal(out, want[0]) and torch.equal(lse, want[1])


@pytest.mark.gpu
def test_a_handler_of_the_callers_own_is_not_recorded(gpu):
    """The plug-in surface: a plan with an instruction whose handler is not this package's runs
    through the handlers on every pass."""
    from dcp_amd.core.instructions import AttnInstr, AttnReductionInstr, MemcpyInstr
    from dcp_amd.runtime.flash_attention import executor as module

    case = make_case(**CASE)
    ex = module.AttentionExecutor(fw_exec_plan=case["fw"], bw_exec_plan=case["bw"], node_id=0, local_device_id=0,
                                  n_devices_per_node=1, n_nodes=1, n_heads_per_block=2, head_dim=128)
    seen = []
    ex.register_handler(MemcpyInstr, module._handle_memcpy)
    ex.register_handler(AttnInstr, lambda e, i: (seen.append(e.instr_index), module._handle_attn(e, i)))
    ex.register_handler(AttnReductionInstr, module._handle_reduction)
    for kind, prep in ((MemcpyInstr, module._prepare_memcpy), (AttnInstr, module._prepare_attn),
                       (AttnReductionInstr, module._prepare_reduction)):
        ex.register_prep_handler(kind, prep)
    ex.prepare(forward=True)
    q, kv = case["layout"].to_local_q(case["q"]).cuda(), case["layout"].to_local_kv(case["kv"]).cuda()
    a, b = ex.forward(q, kv), ex.forward(q, kv)
    assert len(seen) == 4 and ex._recorded is None  # two attention instructions, two passes
    assert torch.equal(a[0], b[0])
