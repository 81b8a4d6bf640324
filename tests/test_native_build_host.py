"""The extension behind the native front end belongs to one torch and one Python: it is built again when either changes, and one that
was built for others, or is missing, is not used -- the wrappers then go their own way, with a warning."""
import importlib.util
import os
import warnings

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture
def build(tmp_path, monkeypatch):
    """build.py with its outputs in a folder of the test and a compiler that only counts"""
    spec = importlib.util.spec_from_file_location("_build_under_test", os.path.join(ROOT, "g-core-gh_amd", "build.py"))
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    b.OBJ, b.NATIVE, b.compiled = str(tmp_path), str(tmp_path / "_lowp_native.so"), []

    def run(cmd, **kw):
        b.compiled.append(cmd)
        open(b.NATIVE, "w").close()
        return type("R", (), {"returncode": 0, "stderr": ""})

    monkeypatch.setattr(b.subprocess, "run", run)
    return b


def test_another_torch_or_python_builds_it_again(build, monkeypatch):
    import sysconfig
    import torch
    build._build_native(False)
    build._build_native(False)
    assert len(build.compiled) == 1
    monkeypatch.setattr(torch.version, "git_version", "0" * 40)
    build._build_native(False)
    build._build_native(False)
    assert len(build.compiled) == 2
    real = sysconfig.get_config_var
    monkeypatch.setattr(sysconfig, "get_config_var", lambda n: "cpython-399" if n == "SOABI" else real(n))
    build._build_native(False)
    assert len(build.compiled) == 3 and any("cpython-399" in a for a in build.compiled[-1])
    monkeypatch.undo()


def test_the_built_extension_is_for_this_torch():
    from gcore_lowp import _native
    assert _native._load().built_for == _native.built_for()


@pytest.mark.parametrize("why", ["missing", "another torch", "not loadable"])
def test_an_extension_for_others_is_not_used(why, tmp_path, monkeypatch):
    from gcore_lowp import _native
    if why == "missing":
        monkeypatch.setattr(_native, "PATH", str(tmp_path / "none.so"))
    elif why == "not loadable":
        (tmp_path / "bad.so").write_bytes(b"not a library")
        monkeypatch.setattr(_native, "PATH", str(tmp_path / "bad.so"))
    else:
        monkeypatch.setattr(_native.torch.version, "git_version", "0" * 40)
    fast = _native._Fast()
    with pytest.warns(RuntimeWarning, match="build it with"):
        assert fast.gemm(None, None, None, None, 0) is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert fast.quant_fp8() is None and fast.dequant() is None and fast.fp4_to_fp8() is None
    with pytest.raises(AttributeError):
        fast.other
