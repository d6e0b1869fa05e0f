"""The native plan analysis is an optional part of the build, for this Python alone (CPU)."""

import importlib.machinery

import pytest

from dcp_amd import build


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
