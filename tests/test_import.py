"""The package works without the extension with the binding's fast calls, which
is built for one Python."""
import glob
import os
import subprocess
import sys
import sysconfig
import types

import pytest

import vortx_amd
from vortx_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _python(code):
    return subprocess.run([sys.executable, "-W", "always", "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=120)


def test_import_without_the_extension():
    r = _python("import sys; sys.modules['vortx_amd._pycall'] = None\n"
                "import vortx_amd as vx\n"
                "assert vx.TensorLayout.contiguous([2, 3]).is_contiguous()\n"
                "print(vx.layout_extent(vx.TensorLayout.contiguous([2, 3])))")
    assert r.returncode == 0, r.stderr
    assert r.stdout.split() == ["6"]
    assert "slower ctypes path" in r.stderr


def test_the_extension_is_named_for_its_python():
    built = glob.glob(os.path.join(os.path.dirname(vortx_amd.__file__), "_pycall*.so"))
    assert built == [build.PYCALL] and built[0].endswith(sysconfig.get_config_var("EXT_SUFFIX"))


@pytest.mark.gpu
def test_calls_without_the_extension(gemm, monkeypatch):
    import torch
    a, b = torch.randn(70, 96, device="cuda"), torch.randn(96, 80, device="cuda")
    want, got = torch.empty(70, 80, device="cuda"), torch.empty(70, 80, device="cuda")
    gemm.dispatch(want, a, b)
    monkeypatch.setattr(vortx_amd, "_pycall", types.SimpleNamespace(gemm=lambda *args: None))
    gemm.dispatch(got, a, b)
    assert torch.equal(got, want)
