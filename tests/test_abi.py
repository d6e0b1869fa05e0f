"""The C-ABI library: it loads, exports every symbol include/dcp_hip.h declares,
and rejects bad arguments before launching anything (no GPU needed: only the
argument checks run here)."""

import ctypes
import re
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def lib():
    from dcp_amd import _lib

    if not _lib.LIB_PATH.exists():
        from dcp_amd import build

        build.build(verbose=False)
    return _lib.load()


def _declared_symbols():
    text = (ROOT / "include" / "dcp_hip.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(dcp_[a-z_0-9]+)\s*\(", text)))


def test_header_and_library_agree(lib):
    from dcp_amd import _lib

    declared = _declared_symbols()
    assert len(declared) >= 12
    for name in declared:
        assert hasattr(lib, name), f"{name} is declared in dcp_hip.h but not exported"
    assert sorted(_lib.SIGNATURES) == declared, "ctypes signatures and header differ"


def test_version_and_error_string(lib):
    assert lib.dcp_version() >= 100
    assert isinstance(lib.dcp_last_error(), bytes)


def test_argument_errors_are_reported_without_a_launch(lib):
    from dcp_amd import _lib

    with pytest.raises(AssertionError, match="unsupported element size"):
        _lib.call("dcp_fused_copy_varlen", 0, 0, 0, 0, 0, 0, 0, 1, 16, 3, 0)
    with pytest.raises(AssertionError, match="Too many blocks"):
        _lib.call("dcp_update_out_lse", 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 64, 1, 1, 1, 1, 1, 1, 64, 128, 0, 0)
    with pytest.raises(ValueError, match="Unsupported dtype"):
        _lib.call("dcp_blockwise_sum", 0, 0, 0, 0, 0, 0, 0, 0, 1, 1, 128, 7, 0)
    with pytest.raises(ValueError, match="head_dim"):
        _lib.call("dcp_attn_fwd", *([0] * 8), 1, 0, 0, 0, 0, 1, 1, 64, 64, 1, 1, 96, 0, 0, 1, 1.0, 0, 0, 0, 0)
    with pytest.raises(ValueError, match="bf16 and fp16"):
        _lib.call("dcp_attn_fwd", *([0] * 8), 1, 0, 0, 0, 0, 1, 1, 64, 64, 1, 1, 128, 0, 0, 1, 1.0, 2, 0, 0, 0)
    # empty problems are accepted and launch nothing
    _lib.call("dcp_fused_copy_varlen", 0, 0, 0, 0, 0, 0, 0, 0, 16, 2, 0)
    _lib.call("dcp_attn_fwd", *([0] * 8), 1, 0, 0, 0, 0, 0, 1, 0, 64, 1, 1, 128, 0, 0, 1, 1.0, 0, 0, 0, 0)
    assert lib.dcp_attn_fwd_workspace_bytes() >= 9 * 4
    assert lib.dcp_attn_bwd_workspace_bytes(2, 128, 64, 4, 128) >= 128 * 4 * 4 + 2 * 8 * 4


def _items_call(items=16, n_items=1, one_each=0, splits=0, n_splits=0, n_partials=0, partials=0, partials_bytes=0,
                workspace=16, workspace_bytes=64):
    """One row of 64-token blocks; the addresses are not read before the arguments have been checked."""
    from dcp_amd import _lib

    _lib.call("dcp_attn_fwd_items", *([16] * 8), 1, *([16] * 3), 0, 1, 1, 64, 64, 1, 1, 64, 64 * 64, 64, 64 * 64, 64 * 64, 64, 64, 0, 1.0, 0,
              workspace, workspace_bytes, items, n_items, one_each, splits, n_splits, n_partials, partials, partials_bytes, 0)


@pytest.mark.parametrize("wrong,message", [
    (dict(items=24), "not 16-byte aligned"),
    (dict(n_items=0), "no items"),
    (dict(n_items=-1), "no items"),
    (dict(items=0), "no table of items"),
    (dict(items=0, n_items=0, splits=16, n_splits=1, n_partials=2, partials=16, partials_bytes=1 << 20), "no table of items"),
    (dict(n_splits=1, n_partials=1), "do not fit"),
    (dict(n_splits=2, n_partials=4), "do not fit"),
    (dict(n_splits=-1), "do not fit"),
    (dict(n_splits=1, n_partials=2), "partials are missing"),
    (dict(splits=16, n_splits=1, n_partials=2, partials=24, partials_bytes=1 << 20), "partials are missing"),
    (dict(splits=16, n_splits=1, n_partials=2, partials=16, partials_bytes=2 * 128 * 66 * 4 - 1), "partials are missing"),
    (dict(workspace=0), "workspace"),
    (dict(workspace=0, one_each=1), "workspace"),
    (dict(workspace_bytes=63, one_each=1), "workspace"),
])
def test_tables_of_items_that_are_refused(lib, wrong, message):
    with pytest.raises(AssertionError, match=message):
        _items_call(**wrong)


def test_sequences_that_are_refused(lib):
    from dcp_amd import _lib

    recording = _lib.Recording()
    assert recording.begin()
    _lib.call("dcp_fused_copy_varlen", 0, 0, 0, 0, 0, 0, 0, 0, 16, 2, 0)  # (nothing to copy: returns before it launches)
    recording.end()
    run = dict(kind=_lib.Sequence.RUN, list=recording._list, end=1)

    def sequence(*ops):
        _lib.call("dcp_sequence_run", (_lib._SequenceOp * len(ops))(*(_lib._SequenceOp(**op) for op in ops)), len(ops), 0)

    sequence()
    _lib.call("dcp_sequence_run", None, 0, 0)
    sequence(run, dict(run, begin=1))
    for ops, message in [
        ([dict(run, list=None)], "null list"),
        ([dict(run, end=2)], "calls 0 to 2 of 1"),
        ([dict(run, begin=-1)], "calls -1 to 1 of 1"),
        ([run, dict(kind=3, event=16)], "operation 1 is of kind 3"),
        ([dict(kind=-1, event=16)], "operation 0 is of kind -1"),
        ([dict(kind=_lib.Sequence.RECORD)], "operation 0 is of kind 1, event"),
        ([run, run, dict(kind=_lib.Sequence.WAIT)], "operation 2 is of kind 2, event"),
    ]:
        with pytest.raises(AssertionError, match=message):
            sequence(*ops)
    for n_ops in (1, -1):
        with pytest.raises(AssertionError, match="no operations"):
            _lib.call("dcp_sequence_run", None, n_ops, 0)


def test_workspaces_have_the_sizes_callers_know(lib):
    """A caller may have its buffers before it asks, for the backward two floats per (query, head), a hull of
    32 bytes per 64-query tile, each rounded up to 256 bytes, and 256 bytes of counters.  A problem
    that just fills the static entry point's scratch stays one."""
    up = lambda n: -(-n // 256) * 256
    for batch, bs, heads in ((1, 64, 1), (3, 128, 5), (508, 1024, 8)):
        total_q = batch * bs
        want = 2 * up(total_q * heads * 4) + up(batch * -(-bs // 64) * 32) + 256
        assert lib.dcp_attn_bwd_workspace_bytes(batch, total_q, bs, heads, 64) == want
    # 8 heads, 64-token rows: (64 * 64 + 32) bytes a row and the counters
    rows = ((32 << 20) - 256) // (64 * 8 * 8 + 32) // 8 * 8
    assert (32 << 20) - 8 * (64 * 8 * 8 + 32) < lib.dcp_attn_bwd_workspace_bytes(rows, rows * 64, 64, 8, 64) <= 32 << 20


def test_backward_selection_and_its_workspace_size(lib):
    """dcp_attn_bwd_select returns the previous setting and only sets a known mode; the workspace the
    selected backward needs: the recomputing one the small scratch whatever the key count, the one
    that keeps dS in memory 4 KiB per (64-key tile, head, 32-query chunk) on top of it, with one tile
    more per row than total_kv / 64 and two spare pieces."""
    before = lib.dcp_attn_bwd_select(0)
    try:
        assert lib.dcp_attn_bwd_select(-1) == 0 and lib.dcp_attn_bwd_select(77) == 0 and lib.dcp_attn_bwd_select(-1) == 0
        batch, total_q, total_kv, bs, heads, d = 6, 6 * 256, 6 * 1024 + 5 * 256, 256, 4, 128
        base = lib.dcp_attn_bwd_workspace_bytes(batch, total_q, bs, heads, d)
        assert lib.dcp_attn_bwd_workspace_bytes_kv(batch, total_q, total_kv, bs, heads, d) == base
        assert lib.dcp_attn_bwd_select(2) == 0
        pieces = (total_kv // 64 + batch + 1) * heads * (bs // 32) + 2
        assert lib.dcp_attn_bwd_workspace_bytes_kv(batch, total_q, total_kv, bs, heads, d) == base + pieces * 4096
        assert lib.dcp_attn_bwd_workspace_bytes_kv(batch, total_q, 0, bs, heads, d) == base, "no key count: nothing to keep"
        assert lib.dcp_attn_bwd_workspace_bytes(batch, total_q, bs, heads, d) == base
    finally:
        lib.dcp_attn_bwd_select(before)


def test_profile_report_is_empty_when_disabled(lib):
    from dcp_amd import _lib

    assert _lib.profile_report() == {}
