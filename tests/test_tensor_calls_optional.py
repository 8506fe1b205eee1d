"""The per-step calls on tensors (_kvhtorch) are built against one PyTorch: with another one, or not built at
all, the library loads all the same and HipAttention's methods do without them, with a warning."""

from __future__ import annotations

import subprocess
import sys
import textwrap
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


def _run(setup: str) -> str:
    code = textwrap.dedent("""
        import sys, types, warnings
        import torch
        import kvserve_amd
        from kvserve_amd import _lib
        {setup}
        with warnings.catch_warnings(record=True) as caught:
            warnings.simplefilter("always")
            _lib.load()
            _lib.load()
        print("fast", _lib.fast() is not None, "calls", _lib.calls() is not None,
              "warned", sum("_kvhtorch" in str(w.message) for w in caught))
    """).format(setup=setup)
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT)
    assert res.returncode == 0, res.stderr
    return res.stdout.strip()


def _gpu_build() -> bool:
    import torch

    return hasattr(torch._C, "_cuda_getCurrentRawStream")


def test_built_for_this_pytorch():
    if not _gpu_build():
        pytest.skip("this PyTorch hands out no stream handles")
    assert _run("") == "fast True calls True warned 0"


def test_not_built():
    n = int(_gpu_build())
    assert _run("sys.modules['kvserve_amd._kvhtorch'] = None") == f"fast True calls False warned {n}"


@pytest.mark.parametrize("version", ["'0.0.0'", "torch.__version__ + 'x'", None])
def test_built_for_another_pytorch(version):
    # a module of another build: never bound, whatever it is (None: one that does not name its PyTorch)
    setup = "m = types.ModuleType('kvserve_amd._kvhtorch'); m.bind = lambda *a: sys.exit('bound'); "
    setup += f"m.torch_version = {version}; " if version else ""
    setup += "sys.modules[m.__name__] = kvserve_amd._kvhtorch = m"
    assert _run(setup) == f"fast True calls False warned {int(_gpu_build())}"
