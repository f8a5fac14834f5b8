"""Which binding module is built and loaded: one that was built for another torch or another interface of the library, or is not there,
is left alone with a warning, and built again when asked.  No GPU."""
import importlib.util
import os
import subprocess
import sys
import types

import pytest
import torch

PKG_ROOT = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "3d-deformable-attention_amd")
HERE = f"{torch.__version__} {torch.version.git_version}"


def _other(built_for, abi):
    module = types.ModuleType("dfa3D._binding")
    module.built_for = lambda: (built_for, abi)
    module.bind = lambda table: pytest.fail("bound all the same")
    return module


@pytest.mark.parametrize("module", [None, _other("2.9.0 abc", 9), _other(HERE, 8), types.ModuleType("dfa3D._binding")],
                         ids=["missing", "other torch", "other ABI", "nameless"])
def test_a_module_that_does_not_fit(monkeypatch, module):
    from dfa3D import _ext, _lib
    from dfa3D.modules import projection
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "_binding", None)
    monkeypatch.setitem(sys.modules, "dfa3D._binding", module)
    with pytest.warns(RuntimeWarning, match="ctypes"):
        handle = _lib.lib()
    assert handle.dfa3d_abi_version() == _lib.ABI_VERSION and _lib.binding() is None
    on_gpu = types.SimpleNamespace(is_cuda=True)
    assert _ext._here(on_gpu) is None and projection._sum_of_products((on_gpu, on_gpu)) is None


def test_the_module_that_was_built_here():
    from dfa3D import _lib
    assert _lib.lib() is not None and _lib.binding().built_for() == (HERE, _lib.ABI_VERSION)


def test_built_again_for_another_torch(monkeypatch, tmp_path, capsys):
    spec = importlib.util.spec_from_file_location("dfa3d_build_for_test", os.path.join(PKG_ROOT, "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    target = tmp_path / "_binding.so"
    monkeypatch.setattr(build, "BINDING", str(target))
    monkeypatch.setattr(build, "BINDING_STAMP", str(tmp_path / "stamps" / "built_for"))
    ran = []

    def run(cmd, verbose):
        ran.append(cmd)
        target.write_bytes(b"")
    monkeypatch.setattr(build, "_run", run)
    assert build._build_binding(False, False) and len(ran) == 1
    assert build._build_binding(False, False) and len(ran) == 1             # up to date
    monkeypatch.setattr(torch, "__version__", "2.99.0")
    assert build._build_binding(False, False) and len(ran) == 2 and any("2.99.0" in a for a in ran[1])

    def fail(cmd, verbose):
        raise subprocess.CalledProcessError(1, cmd)
    monkeypatch.setattr(build, "_run", fail)
    assert not build._build_binding(True, False) and not target.exists()    # not left behind for another torch to load
    assert "ctypes" in capsys.readouterr().err
