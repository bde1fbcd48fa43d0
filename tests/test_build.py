"""Building the library and the module beside it: what a build leaves behind.  No compiler runs here."""
import subprocess
from types import SimpleNamespace

import pytest

from gesso_amd.errors import KernelError
from gesso_amd.kernels import build


@pytest.fixture
def tools(tmp_path, monkeypatch):
    """An earlier build's library, module and digest in the only folder that builds go to, and tools that write what they are asked
    for (``fails``: a word in the command that ends with an error)."""
    told = SimpleNamespace(folder=tmp_path, fails=None)
    monkeypatch.setattr(build, "_lib_dirs", lambda: [str(tmp_path)])
    monkeypatch.setattr(build, "_hipcc", lambda: "hipcc")
    monkeypatch.setattr(build, "_cxx", lambda: "c++")
    monkeypatch.setattr(build, "sources", lambda: ["one.hip", "two.hip"])
    for name in ("libgesso_hip.so", "gesso_host.so", "libgesso_hip.so.digest"):
        (tmp_path / name).write_text("earlier")

    def run(cmd, **kw):
        if told.fails is not None and any(told.fails in c for c in cmd) and (told.fails != "-shared" or cmd[0] == "hipcc"):
            return subprocess.CompletedProcess(cmd, 1, "no")
        with open(cmd[cmd.index("-o") + 1], "w") as f:
            f.write("new")
        return subprocess.CompletedProcess(cmd, 0, "")

    monkeypatch.setattr(build.subprocess, "run", run)
    return told


def _held(folder):
    return {f.name: f.read_text() for f in folder.iterdir() if f.is_file()}


@pytest.mark.parametrize("fails", ["two.hip", "host.cpp", "-shared"])
def test_a_build_that_fails_leaves_library_and_module_as_they_were(tools, fails):
    before = _held(tools.folder)
    tools.fails = fails
    with pytest.raises(KernelError):
        build.build(verbose=False)
    assert _held(tools.folder) == before


def test_a_build_replaces_library_and_module_together(tools):
    path = build.build(verbose=False)
    assert _held(tools.folder) == {"libgesso_hip.so": "new", "gesso_host.so": "new", "libgesso_hip.so.digest": build._digest()}
    assert build.find_built() == path


@pytest.mark.parametrize("flags", ["FLAGS", "LINK", "HOST_FLAGS", "HOST_LINK"])
def test_other_flags_are_another_build(tools, monkeypatch, flags):
    build.build(verbose=False)
    assert build.find_built() is not None
    monkeypatch.setattr(build, flags, getattr(build, flags) + ["-g"])
    assert build.find_built() is None


def test_a_build_with_nothing_to_compile_the_module_with_is_one_without_it(tools, monkeypatch):
    """The kernels need hipcc alone: without a C++ compiler or Python's headers the earlier module goes, and every call is made
    from Python."""
    from gesso_amd.kernels import ops
    for lacks in ("_cxx", "_HOST_INCLUDE"):
        with monkeypatch.context() as m:
            m.setattr(build, lacks, (lambda: None) if lacks == "_cxx" else [str(tools.folder)] * 3)
            assert build.build(verbose=False) == build.find_built()
            assert not (tools.folder / "gesso_host.so").exists() and (tools.folder / "libgesso_hip.so").read_text() == "new"
            m.setattr(build, "load", lambda: SimpleNamespace(_name=build.find_built()))
            m.setattr(build, "_host", None)
            m.setattr(ops, "_host", None)
            assert build.load_host() is None and ops._native().add_rmsnorm(1, 2) is False
    assert build.build(force=False, verbose=False) == build.find_built() and not (tools.folder / "gesso_host.so").exists()
    build.build(verbose=False)
    assert (tools.folder / "gesso_host.so").exists()
    (tools.folder / "gesso_host.so").unlink()                   # (gone, and not by the build's own account)
    assert build.find_built() is None
