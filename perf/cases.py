"""The workloads this repository's performance is measured on, through its public entry points.

Six kinds of call, each over the range of sizes it meets in use:

* ``forward`` / ``backward``: one prepared plan executed by an ``AttentionExecutor`` -- what the
  micro-benchmark of the reference times (``benchmark/microbenchmark/benchmark_attention.py:976-1021``);
* ``step``: a forward and a backward plan, one after the other, as ``bench.py`` runs them;
* ``iteration``: one training iteration's attention through ``DCPAttention``.  DCP plans every
  batch anew, so the executor, its buffers and its argument tables are made for every iteration
  (``benchmark/mlm/monkey_patch.py:213-260``);
* ``exchange``: a forward and a backward of several devices that share the GPU and send each other blocks;
* ``gather`` / ``merge`` / ``sum``: the block operators of ``dcp_amd.ops.fused_ops`` on their own.

A case holds numbers and names only; sequence lengths follow from its ``lengths_seed``.
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

from dcp_amd.core.instructions import BufferType
from dcp_amd.ops.fused_ops import (
    flash_attn_update_out_lse,
    fused_blockwise_sum,
    fused_copy_bf16_varlen,
    fused_copy_fp16_varlen,
    fused_copy_fp32_varlen,
)
from dcp_amd.runtime.flash_attention.executor import DCPAttention, get_executor
from dcp_amd.runtime.flash_attention.fabric import LocalFabric, execute_together
from dcp_amd.runtime.flash_attention.multi_device import build_staged_multi_device_plans
from dcp_amd.runtime.flash_attention.single_device import build_single_device_plans
from dcp_amd.runtime.flash_attention.utils import MASK_FNS, count_attended_pairs

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
COPY = {"bf16": fused_copy_bf16_varlen, "fp16": fused_copy_fp16_varlen, "fp32": fused_copy_fp32_varlen}
ATTENTION_KINDS = ("forward", "backward", "step", "iteration", "exchange")


def _attention(kind, name=None, **changes):
    case = dict(kind=kind, tokens=65536, median=4096, longest=32768, lengths_seed=0, mask="causal", block_size=1024,
                heads=32, kv_heads=8, head_dim=128, head_block=4, partials=1, dtype="bf16")
    case.update(changes)
    if name is not None:
        case["name"] = name
    return case


def _blocks(kind, name=None, **changes):
    case = dict(kind=kind, tokens=262144, heads=32, head_dim=128, block_size=512, sources=1, ragged=False, dtype="bf16")
    case.update(changes)
    if name is not None:
        case["name"] = name
    return case


def listed():
    return [
        # A few short sequences on one device, eight q heads of which four share a kv head: launches and
        # latency count.
        _attention("forward", "forward_short", tokens=1000, median=350, longest=700, block_size=256, heads=8, kv_heads=2),
        # The attention shape of an 8B model on one device: 65536 packed tokens of ragged sequences, causal.
        _attention("forward", "forward_causal_64k"),
        _attention("backward", "backward_causal_64k"),
        # Attention sink plus sliding window over long sequences: two ranges per query, most tiles skipped.
        _attention("step", "step_lambda_128k", tokens=131072, median=16384, longest=65536, mask="lambda"),
        # Long shared contexts with independent continuations; every row's keys come in two partials, so
        # the merge and the dQ sum run (the largest case).
        _attention("step", "step_shared_prefix_96k", tokens=98304, mask="shared_prefix", block_size=512, heads=40,
                   head_block=5, partials=2),
        # The reference's micro-benchmark shape: 8 q and 2 kv heads, 512-token blocks; one head per head
        # block, the finest split of the heads that a plan can have.
        _attention("step", "step_micro_32k", tokens=32768, median=4096, longest=16384, block_size=512, heads=8,
                   kv_heads=2, head_block=1),
        # No grouped queries, head size 64, fp16, short ragged sequences in small blocks.
        _attention("step", "step_fp16_d64_5k", tokens=5120, median=1024, longest=2048, block_size=256, heads=8,
                   kv_heads=8, head_dim=64, head_block=8, dtype="fp16"),
        # One training iteration with a plan of its own: executor, tables, forward and backward.
        _attention("iteration", "iteration_16k", tokens=16384, median=2048, longest=8192, block_size=512, heads=16,
                   kv_heads=4),
        # Four devices' plans (two nodes of two) in two stages, sharing this GPU.
        _attention("exchange", "exchange_4_devices_16k", tokens=16384, median=4096, longest=8192, block_size=512, heads=8,
                   kv_heads=2, devices=4, stages=2),
        # Block movement at the size of a device's whole activations: gather through a permutation of the
        # blocks and scatter back.
        _blocks("gather", "gather_2gib"),
        # Four partial outputs per query block merged, all heads of a token side by side.
        _blocks("merge", "merge_4_of_32k", tokens=32768, sources=4),
        # dQ / dK / dV partials of ragged blocks added up.
        _blocks("sum", "sum_3_of_8k_ragged", tokens=8192, heads=8, sources=3, ragged=True),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(ATTENTION_KINDS + ("step", "gather", "merge", "sum"))
    if kind in ("gather", "merge", "sum"):
        head_dim = rng.choice((64, 128))
        heads = rng.choice((1, 4, 5, 8, 32))
        sources = 1 if kind == "gather" else rng.randint(2, 8)
        tokens = _log_uniform(rng, 512, min(262144, 2**24 // (sources * heads * (head_dim // 64))))
        return _blocks(kind, tokens=tokens, heads=heads, head_dim=head_dim, block_size=rng.choice((256, 512, 1024)),
                       sources=sources, ragged=rng.random() < 0.5,
                       dtype=rng.choice(("bf16", "bf16", "fp16", "fp32")), lengths_seed=rng.randrange(1 << 20))
    heads, kv_heads = rng.choice(((8, 2), (16, 4), (32, 8), (40, 8), (8, 8)))
    group = heads // kv_heads
    tokens = _log_uniform(rng, 512, 16384 if kind == "exchange" else 32768 if kind == "iteration" else 65536)
    longest = min(tokens, _log_uniform(rng, 512, 16384))
    case = _attention(
        kind, tokens=tokens, longest=longest, median=max(64, longest // rng.choice((1, 2, 4, 8))),
        lengths_seed=rng.randrange(1 << 20), mask=rng.choice(("causal", "causal", "lambda", "shared_prefix")),
        block_size=rng.choice((256, 512, 1024)), heads=heads, kv_heads=kv_heads, head_dim=rng.choice((64, 128, 128)),
        head_block=rng.choice((1, group) if group > 1 else (1, heads)), partials=rng.choice((1, 1, 2)),
        dtype=rng.choice(("bf16", "bf16", "fp16")))
    if kind == "exchange":
        case.update(devices=rng.choice((2, 4)), stages=rng.choice((1, 2)), partials=1, block_size=rng.choice((256, 512)))
    return case


# ---------------------------------------------------------------------------
# what a case's numbers stand for
# ---------------------------------------------------------------------------


def _lengths(case):
    """Lognormal sequence lengths that fill exactly ``tokens`` tokens (``bench.py``'s, which clip at
    256 and draw a sequence anew only if what is left would be too short)."""
    rng = np.random.default_rng(case["lengths_seed"])
    total, lo, hi = case["tokens"], min(256, case["longest"] // 2), case["longest"]
    lengths, used = [], 0
    while used < total:
        n = int(np.clip(round(float(np.exp(rng.normal(np.log(case["median"]), 1.0)))), lo, hi))
        if total - used - n < lo:
            n = total - used
            if n > hi:
                n = total - used - lo
        lengths.append(n)
        used += n
    return lengths


def _shared_prefix(case):
    """Samples of one shared context and 4 to 16 continuations of 1/32 to 1/4 of it, until
    ``tokens`` tokens are filled."""
    rng = np.random.default_rng(case["lengths_seed"])
    total = case["tokens"]
    prefix = max(16, min(8192, case["longest"], total // 4))
    seqlens, info = [], []
    while sum(seqlens) < total:
        room = total - sum(seqlens)
        conts = [int(c) for c in rng.integers(prefix // 32 + 1, prefix // 4 + 2, size=int(rng.integers(4, 17)))]
        if room <= prefix + 1:  # too little for another context: lengthen the last sample
            info[-1]["continuations"].append(room)
            seqlens[-1] += room
            break
        kept, room = [], room - prefix
        for c in conts:
            if room > 0:
                kept.append(min(c, room))
                room -= kept[-1]
        info.append(dict(prefix=prefix, continuations=kept))
        seqlens.append(prefix + sum(kept))
    return seqlens, info


@functools.lru_cache(maxsize=64)
def _plans_of(items):
    case = dict(items)
    info, kwargs = None, {}
    if case["mask"] == "shared_prefix":
        seqlens, info = _shared_prefix(case)
    else:
        seqlens = _lengths(case)
    if case["mask"] == "lambda":
        kwargs = dict(n_starting=64, l_pretrain=4096)
    mask = MASK_FNS[case["mask"]](seqlens, seqlens, torch.int32, info, **kwargs)
    args = (seqlens, case["block_size"], case["heads"], case["kv_heads"], case["head_dim"], case["head_block"], mask)
    if case["kind"] == "exchange":
        n_nodes = 2 if case["devices"] == 4 else 1
        fw, bw, _ = build_staged_multi_device_plans(n_nodes, case["devices"] // n_nodes, *args, dtype=DTYPES[case["dtype"]],
                                                    n_stages=case["stages"])
    else:
        fw, bw, _ = build_single_device_plans(*args, dtype=DTYPES[case["dtype"]], n_kv_groups=case["partials"],
                                              kv_split="contiguous", backward=case["kind"] != "forward")
    return fw, bw, count_attended_pairs(mask)


def _plans(case):
    """(forward plan, backward plan, attended pairs) of a case: the planner's work, done once."""
    return _plans_of(tuple(sorted((k, v) for k, v in case.items() if k != "name")))


def work(case):
    elem = 4 if case["dtype"] == "fp32" else 2
    if case["kind"] not in ATTENTION_KINDS:
        per_token = case["heads"] * case["head_dim"] * elem
        rows = int(_block_tokens(case).sum())
        if case["kind"] == "gather":  # packed and scattered back: read and written twice
            return {"bytes": 4 * rows * per_token, "flops": 0}
        n = case["sources"]
        if case["kind"] == "merge":
            return {"bytes": (n + 1) * rows * (per_token + 4 * case["heads"]), "flops": 2 * n * rows * case["heads"] * case["head_dim"]}
        return {"bytes": (n + 1) * rows * per_token, "flops": (n - 1) * rows * case["heads"] * case["head_dim"]}
    # the reference's cost model (dcp/core/cost_model.py:120-127): 4 operations per attended pair, head
    # and element forward, 2.5 times that backward
    pairs = _plans(case)[2]
    q = case["tokens"] * case["heads"] * case["head_dim"] * elem
    kv = 2 * case["tokens"] * case["kv_heads"] * case["head_dim"] * elem
    lse = case["tokens"] * case["heads"] * 4
    per_pair = case["heads"] * case["head_dim"]
    if case["kind"] == "forward":
        return {"bytes": 2 * q + kv + lse, "flops": 4 * pairs * per_pair}
    if case["kind"] == "backward":
        return {"bytes": 4 * q + 2 * kv + lse, "flops": 10 * pairs * per_pair}
    return {"bytes": 4 * q + 2 * kv + lse, "flops": 14 * pairs * per_pair}


def tolerance(case):
    if case["kind"] == "gather":
        return "exact"
    # about four times what the path shows against 64-bit arithmetic: one rounding of the result (bf16
    # 1.7e-3, fp16 2.1e-4, fp32 1.2e-7) for the block operators, that and the rounding of the weights and
    # of dS in attention (bf16 2.1e-3 out, 2.9e-3 dK/dV; fp16 an eighth of that)
    if case["kind"] in ("merge", "sum"):
        return {"rel": {"fp32": 1e-6, "fp16": 9e-4, "bf16": 7e-3}[case["dtype"]]}
    return {"rel": {"fp16": 1.5e-3, "bf16": 1.2e-2}[case["dtype"]]}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _normal(shape, dtype, generator, scale=1.0):
    return (torch.randn(shape, generator=generator, device="cuda") * scale).to(dtype)


def _attention_inputs(plan, dtype, generator):
    """q, kv ~ 0.5 N(0, 1) and dout ~ N(0, 1) in the plan's LOCAL layout."""
    q_shape, kv_shape = (plan.buffer_info[t].buffer_shape for t in (BufferType.LOCAL_Q, BufferType.LOCAL_KV))
    return (_normal(q_shape, dtype, generator, 0.5), _normal(kv_shape, dtype, generator, 0.5),
            _normal(q_shape, dtype, generator))


def _executor(case, fw, bw, forward, fabric=None):
    ex = get_executor(case["head_block"], case["head_dim"], None, fw_exec_plan=fw, bw_exec_plan=bw, fabric=fabric)
    if not forward:
        ex.mode = "Backward"
    ex.prepare(forward=forward)
    return ex


def _give_backward_inputs(ex_b, ex_f, q, kv, dout):
    ex_b.init_forward_input(q, kv)
    ex_b.set_local_out_lse(ex_f.buffers[BufferType.LOCAL_OUT], ex_f.buffers[BufferType.LOCAL_LSE])
    ex_b.init_backward_input(dout)


def _prepare_attention(case, generator):
    fw, bw, _ = _plans(case)
    dtype = DTYPES[case["dtype"]]
    state = dict(case=case, fw=fw, bw=bw)
    if case["kind"] == "exchange":
        n_nodes = 2 if case["devices"] == 4 else 1
        inputs = [_attention_inputs(p, dtype, generator) for p in fw]
        groups = []
        for forward in (True, False):
            fabric = LocalFabric(n_nodes, case["devices"] // n_nodes)
            groups.append([_executor(case, f, b, forward, fabric) for f, b in zip(fw, bw)])
        for ex, (q, kv, _) in zip(groups[0], inputs):
            ex.init_forward_input(q, kv)
        execute_together(groups[0], forward=True)
        for ex_f, ex_b, (q, kv, dout) in zip(*groups, inputs):
            _give_backward_inputs(ex_b, ex_f, q, kv, dout)
        state.update(forward=groups[0], backward=groups[1])
        return state
    q, kv, dout = _attention_inputs(fw, dtype, generator)
    if case["kind"] == "iteration":
        state.update(q=q, kv=kv, dout=dout)
        return state
    ex_f = _executor(case, fw, bw, forward=True)
    ex_f.init_forward_input(q, kv)
    state["forward"] = ex_f
    if case["kind"] != "forward":
        ex_b = _executor(case, fw, bw, forward=False)
        ex_f.execute(fw, is_forward=True)
        _give_backward_inputs(ex_b, ex_f, q, kv, dout)
        state["backward"] = ex_b
        if case["kind"] == "backward":
            del state["forward"]
    return state


def _block_tokens(case):
    """Tokens of every destination block; of ragged ones at least one."""
    n_blocks, last = divmod(case["tokens"], case["block_size"])
    tokens = np.asarray([case["block_size"]] * n_blocks + ([last] if last else []), dtype=np.int64)
    if case["ragged"]:
        rng = np.random.default_rng(case.get("lengths_seed", 0))
        tokens = np.minimum(tokens, rng.integers(1, case["block_size"] + 1, size=len(tokens)))
    return tokens


def _table(values, dtype=torch.int32):
    return torch.as_tensor(np.ascontiguousarray(values), dtype=dtype, device="cuda")


def _prepare_blocks(case, generator, seed):
    dtype = DTYPES[case["dtype"]]
    bs, heads, dim, n_src = case["block_size"], case["heads"], case["head_dim"], case["sources"]
    n_tokens = _block_tokens(case)
    n = len(n_tokens)
    numel = bs * heads * dim
    order = np.random.default_rng(seed).permutation(n * n_src)
    src = _normal((n * n_src, bs, heads, dim), dtype, generator)
    state = dict(case=case, src=src, numel=numel)
    numels, strides = _table(n_tokens * heads * dim), _table([numel] * n)
    pointers = lambda t: _table([t.data_ptr()] * n, torch.int64)
    if case["kind"] == "gather":
        packed, back = torch.zeros_like(src), torch.zeros_like(src)
        here, there = _table(np.arange(n)), _table(order)
        state.update(packed=packed, back=back,
                     gather=(pointers(src), here, strides, pointers(packed), there, strides, numels),
                     scatter=(pointers(packed), there, strides, pointers(back), here, strides, numels))
        return state
    width = 1 << (n_src - 1).bit_length()
    table = np.full((n, width), -1, dtype=np.int64)
    table[:, :n_src] = order.reshape(n, n_src)
    counts = _table([n_src] * n)
    if case["kind"] == "merge":
        lse = torch.rand((heads, n * n_src, bs), generator=generator, device="cuda") * 10 - 5
        starts = np.concatenate(([0], np.cumsum(n_tokens)))
        out = torch.zeros((int(starts[-1]), heads, dim), dtype=dtype, device="cuda")
        out_lse = torch.zeros((heads, int(starts[-1])), device="cuda")
        state.update(out=out, out_lse=out_lse, args=(
            src, out, lse, out_lse, heads, _table(table), _table(starts[:-1]), _table(n_tokens), counts, bs, numel,
            heads * dim, bs, 1, n * n_src * bs, int(starts[-1]), dim, width, 64))
        return state
    out = torch.zeros((n, bs, heads, dim), dtype=dtype, device="cuda")
    state.update(out=out, args=(pointers(src), _table(table), strides, counts, pointers(out), _table(np.arange(n)), strides,
                                numels, dtype, width, numel, 128))
    return state


def prepare(case, seed):
    generator = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] in ATTENTION_KINDS:
        return _prepare_attention(case, generator)
    return _prepare_blocks(case, generator, seed)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "forward":
        return state["forward"].execute(state["fw"], is_forward=True)
    if kind == "backward":
        return state["backward"].execute(state["bw"], is_forward=False)
    if kind == "step":
        return (*state["forward"].execute(state["fw"], is_forward=True),
                *state["backward"].execute(state["bw"], is_forward=False))
    if kind == "iteration":
        q, kv = state["q"].detach().requires_grad_(), state["kv"].detach().requires_grad_()
        executor = get_executor(case["head_block"], case["head_dim"], None, fw_exec_plan=state["fw"], bw_exec_plan=state["bw"])
        executor.prepare(forward=True)
        out = DCPAttention.apply(executor, False, False, q, kv)
        dq, dkv = torch.autograd.grad(out, (q, kv), state["dout"])
        return out.detach(), dq, dkv
    if kind == "exchange":
        execute_together(state["forward"], forward=True)
        execute_together(state["backward"], forward=False)
        outputs = []
        for ex_f, ex_b in zip(state["forward"], state["backward"]):
            outputs += [ex_f.buffers[BufferType.LOCAL_OUT], ex_f.buffers[BufferType.LOCAL_LSE],
                        ex_b.buffers[BufferType.LOCAL_dQ], ex_b.buffers[BufferType.LOCAL_dKV]]
        return outputs
    if kind == "gather":
        COPY[case["dtype"]](*state["gather"], state["numel"], 128)
        COPY[case["dtype"]](*state["scatter"], state["numel"], 128)
        return state["packed"], state["back"]
    if kind == "merge":
        flash_attn_update_out_lse(*state["args"])
        return state["out"], state["out_lse"]
    fused_blockwise_sum(*state["args"])
    return state["out"]
