"""``_native.so`` belongs to one torch: built again for another one, and refused by another one."""

import os

import pytest
import torch

from instantmimic_amd import _lib
from instantmimic_amd import build as B


@pytest.fixture
def commands(monkeypatch, tmp_path):
    """build_native() into a temporary folder, with the compiler's command lines recorded."""
    ran = []
    monkeypatch.setattr(B, "NATIVE", str(tmp_path / "_native.so"))
    monkeypatch.setattr(B, "OBJ", str(tmp_path / "_obj"))
    monkeypatch.delenv("IMHIP_REBUILD", raising=False)

    def run(cmd, check):
        ran.append(cmd)
        open(B.NATIVE, "w").close()

    monkeypatch.setattr(B.subprocess, "run", run)
    return ran


def test_built_again_for_another_torch(commands, monkeypatch):
    B.build_native()
    B.build_native()
    assert len(commands) == 1
    os.utime(B.NATIVE, (2e9, 2e9))  # a newer file does not make it the right one
    monkeypatch.setattr(torch, "__version__", "9.9.9")
    B.build_native()
    B.build_native()
    assert len(commands) == 2 and '-DIM_TORCH_VERSION="9.9.9"' in commands[1]
    monkeypatch.setattr(torch.version, "git_version", "another commit")
    B.build_native()
    assert len(commands) == 3
    os.remove(B.NATIVE)
    B.build_native()
    assert len(commands) == 4
    monkeypatch.setenv("IMHIP_REBUILD", "1")
    B.build_native()
    assert len(commands) == 5


def test_a_module_for_another_torch_is_refused(monkeypatch):
    assert _lib.native().torch_version == torch.__version__
    monkeypatch.setattr(_lib, "_native", None)
    monkeypatch.setattr(torch, "__version__", "9.9.9")
    with pytest.raises(RuntimeError, match="built for torch"):
        _lib.native()
