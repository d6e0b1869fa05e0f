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


def test_recording_without_host_memory_throws_nothing_at_a_c_caller(tmp_path):
    import subprocess
    from pathlib import Path

    from dcp_amd import _lib

    root, program = Path(__file__).parent, tmp_path / "record_no_memory"
    lib = Path(_lib.LIB_PATH).parent
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{root.parent / 'include'}", str(root / "abi_host" / "record_no_memory.cpp"), "-o",
                    str(program), f"-L{lib}", "-ldcp_hip", f"-Wl,-rpath,{lib}:/opt/rocm/lib", "-Wl,--allow-shlib-undefined"], check=True)
    ran = subprocess.run([str(program)], capture_output=True, text=True, timeout=60)
    assert ran.returncode == 0 and ran.stdout.strip() == "ok", ran.stdout + ran.stderr


def test_a_recording_keeps_what_its_calls_point_to():
    import weakref

    from dcp_amd.runtime.flash_attention import executor as module

    ex = module.AttentionExecutor.__new__(module.AttentionExecutor)
    memory = [torch.zeros(4) for _ in range(4)]
    ex._args_cache = {0: (memory[0],)}
    ex._dkv_partials, ex._bwd_workspace, ex._fwd_partials = memory[1:]
    alive = [weakref.ref(t) for t in memory]
    recording = ex._recording()
    recording.end()
    ex._args_cache = {}
    ex._dkv_partials = ex._bwd_workspace = ex._fwd_partials = None
    memory.clear()
    assert all(r() is not None for r in alive)
    del recording
    assert all(r() is None for r in alive)


class _Stream:
    """Which pieces of work are over when the next piece on the stream begins."""

    def __init__(self, name, handle=1):
        self.name, self.cuda_stream, self.over, self.gone = name, handle, set(), False

    def work(self, what):
        self.over.add(what)

    def wait_stream(self, other):
        assert not other.gone, f"waits on {other.name}, which has been destroyed"
        self.over |= other.over

    def wait_event(self, event):
        self.over |= event.over


class _Event:
    def record(self, stream):
        self.over = set(stream.over)


def _executor_on_streams(monkeypatch, replay=False):
    """An executor whose passes (unless ``replay``) and copies are marks on streams like these, without a GPU;
    ``use(stream)`` makes a stream the caller's."""
    from dcp_amd.core.executor import HandlerTable
    from dcp_amd.core.instructions import BufferType
    from dcp_amd.runtime.flash_attention import executor as module

    current = [None]
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: current[0])
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "Event", _Event)
    ex = module.AttentionExecutor.__new__(module.AttentionExecutor)
    ex.main_stream = _Stream("main")
    ex.main_stream.device_index = 0
    ex._last_stream = ex._last_pass = ex.cuda_graph = None
    ex._handlers = HandlerTable("Instruction handler")
    ex.streams, ex._recorded_steps, ex._steps_of = {}, {}, (None, ())
    ex.kernel_head_dim = ex.head_dim = 64

    class Buffer:
        def copy_(self, value):
            current[0].work(value)

    ex.buffers = {t: Buffer() for t in (BufferType.LOCAL_Q, BufferType.LOCAL_KV, BufferType.LOCAL_dOUT, BufferType.LOCAL_OUT,
                                        BufferType.LOCAL_LSE, BufferType.LOCAL_dQ, BufferType.LOCAL_dKV)}
    monkeypatch.setattr(module.AttentionExecutor, "init_buffers", lambda self, plan: None)
    if not replay:
        monkeypatch.setattr(ex, "_replay", lambda plan, stream: stream.work(plan) or True)
    return ex, lambda stream: current.__setitem__(0, stream)


@pytest.mark.parametrize("handle", [0, 1])
@pytest.mark.parametrize("then", ["execute", "begin", "inputs", "dout", "out_lse"])
def test_what_follows_a_pass_on_another_stream_waits_for_it(monkeypatch, then, handle):
    """Passes share buffers, so whatever runs kernels on them or writes them waits for the last pass, also if
    that pass was on a stream that is gone by then."""
    ex, use = _executor_on_streams(monkeypatch)
    first, second = _Stream("first", handle), _Stream("second", 2)
    use(first)
    ex.execute("a pass", True)
    first.gone = handle != 0
    use(second)
    {"execute": lambda: ex.execute("another", True), "begin": lambda: ex.begin("another"), "inputs": lambda: ex.init_forward_input("q", "kv"),
     "dout": lambda: ex.init_backward_input("dout"), "out_lse": lambda: ex.set_local_out_lse("out", "lse")}[then]()
    assert "a pass" in (ex.main_stream if then == "begin" else second).over


def _set(name, value):
    return lambda ex: setattr(ex, name, value)


@pytest.mark.parametrize("change", [_set("synchronous", True), _set("logger", object()),
                                    _set("_execute_instruction", lambda instr: None), _set("init_buffers", lambda plan: None)],
                         ids=["synchronous", "logger", "own_instruction_loop", "own_buffers"])
def test_switches_set_after_the_first_pass_are_seen(monkeypatch, change):
    """The recorded calls stand for a pass that is nothing but its handlers."""
    from contextlib import nullcontext
    from types import SimpleNamespace

    ex, use = _executor_on_streams(monkeypatch, replay=True)
    use(_Stream("callers", 0))
    ran = []
    calls = SimpleNamespace(run=lambda *a: ran.append(a))
    ex.synchronous, ex.logger, ex.buffers = False, None, {}
    plan = SimpleNamespace(instructions=["an instruction"])
    ex._recorded, ex._recorded_steps, ex._steps_of = (plan, (), calls, 3), {0: (calls, 2)}, (plan, ())
    handle = ex.main_stream.cuda_stream
    assert ex._replay(plan, ex.main_stream) and ran == [(0, 3, handle)]
    ex.begin(plan)
    ex.step(0)
    assert ran == [(0, 3, handle), (0, 2, handle)]
    change(ex)
    assert not ex._replay(plan, ex.main_stream)
    seen = []
    ex.begin(plan)
    monkeypatch.setattr(torch.cuda, "stream", lambda stream: nullcontext())
    monkeypatch.setattr(ex, "_execute_instruction", seen.append)
    ex.step(0)
    assert seen == ["an instruction"] and len(ran) == 2


def test_a_recorded_step_runs_on_the_executors_device(monkeypatch):
    """Whatever device is the caller's current one."""
    from contextlib import contextmanager
    from types import SimpleNamespace

    current, ran_on = [1], []

    @contextmanager
    def device(index):
        before, current[0] = current[0], index
        yield
        current[0] = before

    ex, use = _executor_on_streams(monkeypatch)
    monkeypatch.setattr(torch.cuda, "device", device)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: current[0])
    use(_Stream("callers", 0))
    ex.synchronous, ex.logger, ex.buffers, ex._steps_of = False, None, {}, ("plan", ())
    ex._recorded_steps = {0: (SimpleNamespace(run=lambda *a: ran_on.append(current[0])), 1)}
    ex.begin("plan")
    ex.step(0)
    assert ran_on == [0] and current == [1]


def test_a_pass_in_steps_is_a_pass(monkeypatch):
    ex, use = _executor_on_streams(monkeypatch)
    first, second = _Stream("first"), _Stream("second", 2)
    use(first)
    ex.begin("a plan")
    ex.main_stream.work("a step")
    ex.finish()
    first.gone = True
    use(second)
    ex.execute("another", True)
    assert "a step" in second.over


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


@pytest.mark.gpu
@pytest.mark.parametrize("inputs_first", [False, True])
def test_inputs_of_a_pass_on_another_stream_wait_for_the_last_one(gpu, inputs_first):
    """A pass is held up on one stream while another stream gives the executor new inputs and runs it."""
    case, other = make_case(**CASE), make_case(**CASE, seed=3)
    ex = _executors(case)
    inputs = [(c["layout"].to_local_q(c["q"]).cuda(), c["layout"].to_local_kv(c["kv"]).cuda()) for c in (case, other)]
    want = [ex.forward(*x) for x in inputs]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    with torch.cuda.stream(streams[0]):
        if inputs_first:
            ex.init_forward_input(*inputs[0])
        torch.cuda._sleep(20_000_000)
        got = [ex.forward(*inputs[0])] if not inputs_first else [tuple(t.clone() for t in ex.execute(case["fw"], True))]
    with torch.cuda.stream(streams[1]):
        got.append(ex.forward(*inputs[1]))
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for g, w in zip(got, want) for a, b in zip(g, w))


@pytest.mark.gpu
def test_a_pass_in_steps_waits_for_the_last_pass(gpu):
    from dcp_amd.runtime.flash_attention.fabric import execute_together

    case = make_case(**CASE)
    ex = _executors(case)
    want = ex.forward(case["layout"].to_local_q(case["q"]).cuda(), case["layout"].to_local_kv(case["kv"]).cuda())
    streams = [torch.cuda.Stream() for _ in range(2)]
    for turn in range(2):  # (the second time the steps are recorded)
        torch.cuda.synchronize()
        with torch.cuda.stream(streams[0]):
            torch.cuda._sleep(20_000_000)
            ex.execute(case["fw"], True)
            marker = torch.cuda.Event()
            marker.record()
        with torch.cuda.stream(streams[1]):
            execute_together([ex])
            out = ex.buffers["LocalOut"].clone()
            done = torch.cuda.Event()
            done.record()
        done.synchronize()
        assert marker.query()
        assert torch.equal(out, want[0])


@pytest.mark.gpu
def test_a_synchronous_executor_synchronises_after_the_first_pass_too(gpu):
    case = make_case(**CASE)
    ex = _executors(case)
    q, kv = case["layout"].to_local_q(case["q"]).cuda(), case["layout"].to_local_kv(case["kv"]).cuda()
    want = ex.forward(q, kv)
    assert ex._recorded is not None
    waits = []
    ex.register_synchronization_handler(lambda: (waits.append(1), torch.cuda.synchronize()))
    ex.synchronous = True
    got = ex.forward(q, kv)
    assert len(waits) == len(case["fw"].instructions)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
