"""The build: the native plan analysis is an optional part of it, for this Python alone; what the compiler made of the
kernels (CPU)."""

import importlib.machinery
import re
import struct
import subprocess
from pathlib import Path

import pytest
import yaml

from dcp_amd import build

READELF, OBJDUMP = (Path(build.HIPCC).resolve().parents[1] / "lib" / "llvm" / "bin" / tool for tool in ("llvm-readelf", "llvm-objdump"))


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


def _code_objects(library: Path):
    """The device code in a library."""
    data, magic, found = library.read_bytes(), b"__CLANG_OFFLOAD_BUNDLE__", []
    at = data.find(magic)
    while at >= 0:
        n, entry = struct.unpack_from("<Q", data, at + len(magic))[0], at + len(magic) + 8
        for _ in range(n):
            offset, size, name_size = struct.unpack_from("<3Q", data, entry)
            if size and data[entry + 24 : entry + 27] == b"hip":
                found.append(data[at + offset : at + offset + size])
            entry += 24 + name_size
        at = data.find(magic, at + 1)
    return found


def _kernels(library: Path, where: Path):
    """What the code objects in a library say of their kernels."""
    found = {}
    for code in _code_objects(library):
        (where / "code_object").write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(where / "code_object")], capture_output=True, text=True, check=True).stdout
        metadata = yaml.safe_load(notes[notes.index("---") : notes.index("\n...")])
        found.update({k[".name"]: k for k in metadata["amdhsa.kernels"]})
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


def _instructions(library: Path, kernel: str, where: Path):
    """The mnemonics of the kernels whose names hold ``kernel``, each kernel's in order."""
    objects, found = _code_objects(library), {}
    for i, code in enumerate(objects):
        (where / f"{i}").write_bytes(code)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(where / f"{i}")], capture_output=True, text=True, check=True).stdout
        for name, body in re.findall(r"^<(\S+)>:\n((?:.+\n)*)", text, flags=re.M):
            if kernel in name:
                found[name] = [line.split()[0] for line in body.splitlines() if line.strip()]
    return found


def test_the_probe_has_the_instructions_of_the_dkv_kernel(tmp_path):
    """bench.py divides the dK/dV kernel's rate by that of a probe with its instruction mix: matrix products of the same
    form, and between them, not before or after, the vector instructions, exponentials and LDS reads of a sub-step without a
    mask."""
    if not (build.LIB_PATH.exists() and build.PROBES_LIB.exists()):
        build.build(verbose=False)
        build.build_bench_probes(verbose=False)
    products = lambda body: [i for i in body if i.startswith("v_mfma")]
    kernels = _instructions(build.LIB_PATH, "attn_bwd_dkv_kernelILi0ELi128ELb1E", tmp_path)
    assert len(kernels) == 1 and all({*products(body)} == {"v_mfma_f32_16x16x32_bf16"} for body in kernels.values())
    (body,) = _instructions(build.PROBES_LIB, "mfma_mix_probe_kernelILb1E", tmp_path).values()
    at = [i for i, name in enumerate(body) if name == "v_mfma_f32_16x16x32_bf16"]
    assert len(at) == len(products(body)) == 64
    between = [body[a + 1 : b] for a, b in zip(at, at[1:] + [len(body)])]
    count = lambda some, *names: sum(i.startswith(names) for i in some)
    for names, total in ((("v_fma",), 72), (("v_exp",), 16), (("ds_read_b128",), 22), (("ds_read_b64",), 32)):
        counts = [count(some, *names) for some in between[:-1]]
        assert total - 4 <= sum(counts) <= total and max(counts) <= -(-total // 64) + 2, (names, counts)
