"""The extension module beside the library: built for this torch and this Python, or neither loaded nor left as it is (CPU)."""
import importlib.util
import os

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture
def build_module():
    spec = importlib.util.spec_from_file_location("mase_hip_build_under_test", os.path.join(ROOT, "mase-triton_amd", "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_extension_of_another_torch_is_refused(monkeypatch):
    from mase_hip import _lib

    assert _lib.host().built_for.startswith(f"torch {torch.__version__},")
    monkeypatch.setattr(_lib, "_host", None)
    monkeypatch.setattr(torch, "__version__", "0.0.0+elsewhere")
    with pytest.raises(RuntimeError, match="build it again"):
        _lib.host()
    assert _lib._host is None


def test_extension_is_built_again_for_another_torch(build_module, monkeypatch, tmp_path):
    built = []
    monkeypatch.setattr(build_module, "_stale", lambda target, deps: False)       # every file is newer than its sources
    monkeypatch.setattr(build_module, "build_host", lambda verbose=True: built.append(1))
    stamp = tmp_path / "built_for"
    monkeypatch.setattr(build_module, "HOST_BUILT_FOR", str(stamp))
    for text, builds in ((None, 1), (build_module.host_built_for(), 1), (build_module.host_built_for().replace(torch.__version__, "0.0.0"), 2)):
        if text is not None:
            stamp.write_text(text)
        build_module.build_library(verbose=False)
        assert len(built) == builds
