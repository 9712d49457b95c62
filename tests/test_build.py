"""The build of the library does not depend on the Python operators' host path beside it."""
import os
import stat

import pytest

from phoenix_core_amd import build


@pytest.fixture
def toolchain(tmp_path, monkeypatch):
    """A compiler that only writes its output file; everything is built below tmp_path."""
    hipcc = tmp_path / "hipcc"
    hipcc.write_text("#!/bin/sh\nwhile [ $# -gt 0 ]; do [ \"$1\" = -o ] && echo made > \"$2\"; shift; done; true\n")
    hipcc.chmod(hipcc.stat().st_mode | stat.S_IXUSR)
    csrc = tmp_path / "csrc"
    csrc.mkdir()
    (csrc / "one.hip").write_text("")
    for name, value in (("HERE", tmp_path), ("CSRC", csrc), ("LIB_DIR", tmp_path / "lib"), ("LIB_PATH", tmp_path / "lib" / "lib.so"),
                        ("HOST_PATH", tmp_path / "lib" / "host.so"), ("HIPCC", hipcc)):
        monkeypatch.setattr(build, name, str(value))
    return hipcc


def _no_torch():
    raise ImportError("No module named 'torch'")


@pytest.mark.parametrize("cause", ["compiler fails", "no compiler", "no torch"])
def test_the_library_is_linked_without_the_host_path(cause, toolchain, monkeypatch):
    if cause == "no torch":
        monkeypatch.setattr(build, "_host_command", _no_torch)
    else:
        monkeypatch.setenv("CXX", "false" if cause == "compiler fails" else "/no/such/compiler")
    with pytest.raises(Exception) as raised:
        build.build(verbose=False)
    assert os.path.isfile(build.LIB_PATH) and not os.path.isfile(build.HOST_PATH)
    assert "host path" in str(raised.value)


def test_both_are_built(toolchain, monkeypatch):
    monkeypatch.setenv("CXX", str(toolchain))
    assert build.build(verbose=False) == build.LIB_PATH
    assert os.path.isfile(build.LIB_PATH) and os.path.isfile(build.HOST_PATH)


def test_a_kernel_that_does_not_compile_is_named(toolchain, monkeypatch):
    monkeypatch.setattr(build, "HIPCC", "false")
    monkeypatch.setenv("CXX", "false")
    with pytest.raises(RuntimeError, match="one.hip"):
        build.build(verbose=False)
