"""The build: the native plan analysis is an optional part of it, for this Python alone; what the compiler made of the
kernels (CPU)."""

import importlib.machinery
import struct
import subprocess
from pathlib import Path

import pytest
import yaml

from dcp_amd import build

READELF = Path(build.HIPCC).resolve().parents[1] / "lib" / "llvm" / "bin" / "llvm-readelf"


@pytest.fixture
def elsewhere(monkeypatch, tmp_path):
    """Where it is built to, with what an older build may have left there."""
    monkeypatch.setattr(build, "PLAN_ANALYSIS_LIB", tmp_path / build.PLAN_ANALYSIS_LIB.name)
    (tmp_path / "_plan_analysis.so").write_bytes(b"older")
    build.PLAN_ANALYSIS_LIB.write_bytes(b"older")
    return tmp_path


def test_the_module_is_tagged_and_the_only_one_left(elsewhere):
    suffix = importlib.machinery.EXTENSION_SUFFIXES[0]
    assert "cpython" in suffix and build.build_plan_analysis(verbose=False) == elsewhere / f"_plan_analysis{suffix}"
    assert [f.name for f in elsewhere.iterdir()] == [f"_plan_analysis{suffix}"]
    assert build.PLAN_ANALYSIS_LIB.stat().st_size > 1000


@pytest.mark.parametrize("what", ["compiler", "headers"])
def test_a_build_without(elsewhere, monkeypatch, what):
    if what == "compiler":
        monkeypatch.setenv("CXX", str(elsewhere / "none"))
    else:
        monkeypatch.setattr(build.sysconfig, "get_paths", lambda: dict(include=str(elsewhere)))
    with pytest.warns(RuntimeWarning, match="without the native plan analysis"):
        assert build.build_plan_analysis(verbose=False) is None
    assert list(elsewhere.iterdir()) == []


def _kernels(library: Path, where: Path):
    """What the code objects in a library say of their kernels."""
    data, magic, found = library.read_bytes(), b"__CLANG_OFFLOAD_BUNDLE__", {}
    at = data.find(magic)
    while at >= 0:
        n, entry = struct.unpack_from("<Q", data, at + len(magic))[0], at + len(magic) + 8
        for _ in range(n):
            offset, size, name_size = struct.unpack_from("<3Q", data, entry)
            name = data[entry + 24 : entry + 24 + name_size]
            entry += 24 + name_size
            if name.startswith(b"hip") and size:
                (where / "code_object").write_bytes(data[at + offset : at + offset + size])
                notes = subprocess.run([READELF, "--notes", str(where / "code_object")], capture_output=True, text=True, check=True).stdout
                metadata = yaml.safe_load(notes[notes.index("---") : notes.index("\n...")])
                found.update({k[".name"]: k for k in metadata["amdhsa.kernels"]})
        at = data.find(magic, at + 1)
    return found


def test_no_kernel_spills_vector_registers(tmp_path):
    """A reload from scratch memory waits for every global load in flight, the tiles requested a step ahead among them."""
    if not build.LIB_PATH.exists():
        build.build(verbose=False)
    kernels = _kernels(build.LIB_PATH, tmp_path)
    for name in ("attn_fwd_kernel", "attn_bwd_dkv_kernel", "attn_bwd_dq_kernel", "attn_bwd_dq_ds_kernel", "attn_bwd_fused_kernel"):
        assert sum(name in k for k in kernels) >= 2
    assert {name: k[".private_segment_fixed_size"] for name, k in kernels.items()
            if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]} == {}
