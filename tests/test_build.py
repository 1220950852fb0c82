"""When the host extension is built again."""
import importlib.util
import os
import types

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_host_extension_follows_the_torch_installation(monkeypatch, tmp_path):
    """Built once, then only after its sources or the torch it is linked against have changed."""
    spec = importlib.util.spec_from_file_location("fla_amd_build", os.path.join(ROOT, "flash-linear-attention_amd", "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    path, runs = tmp_path / "_fla_host.so", []
    monkeypatch.setattr(mod, "OBJ_DIR", str(tmp_path))
    monkeypatch.setattr(mod, "HOST_PATH", str(path))

    def run(cmd, **kw):
        runs.append(cmd)
        path.write_text("")
        return types.SimpleNamespace(returncode=0, stdout="", stderr="")

    monkeypatch.setattr(mod.subprocess, "run", run)
    for want in (1, 1):
        mod._build_host(False)
        assert len(runs) == want
    monkeypatch.setattr(torch, "__version__", "0.0.1")
    for want in (2, 2):
        mod._build_host(False)
        assert len(runs) == want
    os.utime(path, (0, 0))
    mod._build_host(False)
    assert len(runs) == 3
