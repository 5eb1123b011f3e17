"""The native host module is optional and belongs to one torch: stale, missing and half-written files."""
import os
import shutil
import warnings

import pytest
import torch


@pytest.fixture
def fresh(monkeypatch, tmp_path):
    """The build and loader modules with an empty folder for the native module and none loaded."""
    from cottention_transformer_amd import _loader, build
    monkeypatch.setattr(build, "HERE", str(tmp_path))
    monkeypatch.setattr(_loader, "_native", None)
    return _loader, build


def test_calls_go_on_in_python_without_it(fresh, monkeypatch):
    """No compiler; a file that cannot be loaded: one warning, and operators that answer as their Python does."""
    loader, build = fresh
    from cottention_transformer_amd import ops

    def no_compiler():
        raise FileNotFoundError("g++")
    monkeypatch.setattr(build, "build_native", no_compiler)
    for broken in (False, True):
        monkeypatch.setattr(loader, "_native", None)
        if broken:
            with open(build.native_path(), "wb") as f:
                f.write(b"not a shared object")
        q = torch.randn(1, 2, 8, 32)
        with pytest.warns(RuntimeWarning, match="native host module"):
            with pytest.raises(RuntimeError, match="must be a CUDA tensor"):
                ops.causal_dot_product(q, q, q)
        with warnings.catch_warnings():
            warnings.simplefilter("error")
            assert loader.native().causal(q, q, q, False) is None and loader.native().decode_block() is None


def test_a_file_of_another_torch_or_source_is_not_taken(fresh, monkeypatch, tmp_path):
    loader, build = fresh
    here = build.native_path()
    assert here == build.native_path() and os.path.dirname(here) == str(tmp_path)
    with monkeypatch.context() as m:
        m.setattr(torch, "__version__", "1.0")
        assert build.native_path() != here
    shutil.copy(os.path.join(build.CSRC, "native.cpp"), tmp_path)
    with open(tmp_path / "native.cpp", "a") as f:
        f.write("// changed\n")
    monkeypatch.setattr(build, "CSRC", str(tmp_path))
    assert build.native_path() != here


def test_outputs_appear_whole(fresh, monkeypatch, tmp_path):
    """Two builds at a time write two files; the final name appears by a rename, and a failed build leaves nothing."""
    loader, build = fresh
    written = []
    path = str(tmp_path / "out.so")

    def compiler(cmd, **kw):
        written.append(cmd[-1])
        if len(written) == 1:  # another build of the same file starts and ends while this one writes
            build._run_to(path, ["cc"], "failed")
        assert not os.path.exists(cmd[-1])
        with open(cmd[-1], "w") as f:
            f.write("whole")
        return type("Done", (), {"returncode": 0, "stdout": ""})
    monkeypatch.setattr(build.subprocess, "run", compiler)
    build._run_to(path, ["cc"], "failed")
    assert len(set(written)) == 2 and path not in written and os.listdir(tmp_path) == ["out.so"]
    assert open(path).read() == "whole"
    monkeypatch.setattr(build.subprocess, "run", lambda cmd, **kw: open(cmd[-1], "w").close() or type(
        "Done", (), {"returncode": 1, "stdout": "error: x"}))
    with pytest.raises(RuntimeError, match="error: x"):
        build._run_to(str(tmp_path / "other.so"), ["cc"], "failed")
    assert os.listdir(tmp_path) == ["out.so"]


def test_the_library_is_built_without_it(fresh, monkeypatch, tmp_path):
    """build() has the kernel library in place before it tries the host module; loading the library builds that alone."""
    loader, build = fresh
    done = []
    monkeypatch.setattr(build, "build_library", lambda *a: done.append("library") or "path")

    def broken():
        done.append("native")
        raise RuntimeError("g++ failed")
    monkeypatch.setattr(build, "build_native", broken)
    with pytest.raises(RuntimeError):
        build.build()
    assert done == ["library", "native"]
    monkeypatch.setattr(loader, "_lib", None)
    monkeypatch.setattr(loader, "lib_path", lambda: str(tmp_path / "none.so"))
    with pytest.raises(OSError):
        loader.lib()
    assert done == ["library", "native", "library"]


def test_old_files_are_removed_by_a_build(fresh, monkeypatch, tmp_path):
    loader, build = fresh
    monkeypatch.setattr(build, "build_library", lambda *a: "path")
    monkeypatch.setattr(build, "build_native", lambda: open(build.native_path(), "w").close() or build.native_path())
    for name in ("_native.so", "_native.0123.so", "other.so"):
        open(tmp_path / name, "w").close()
    build.build()
    assert sorted(os.listdir(tmp_path)) == sorted([os.path.basename(build.native_path()), "other.so"])
