"""What atex_amd/build.py makes of its surroundings, with the compilers stubbed out: the C library does
not depend on torch, and the extension for torch follows the torch it was built for."""
import os
import subprocess

import pytest

from atex_amd import build as B


@pytest.fixture
def stubbed(tmp_path, monkeypatch):
    """build() with its paths under tmp_path; returns (linked libraries, g++ commands)."""
    linked, commands = [], []
    for name in ("OBJ_DIR", "LIB_DIR"):
        monkeypatch.setattr(B, name, str(tmp_path))
    for name in ("LIB_PATH", "BENCH_LIB_PATH", "RESOURCES_PATH", "TORCH_HOST_PATH"):
        monkeypatch.setattr(B, name, str(tmp_path / name))
    monkeypatch.setattr(B, "_compile", lambda src, force, dep_m, bench: str(tmp_path / (src + ".o")))
    monkeypatch.setattr(B, "_link", lambda objs, path, force: linked.append(os.path.basename(path)))

    def run(cmd, **kw):
        commands.append(cmd)
        with open(cmd[cmd.index("-o") + 1], "w") as f:
            f.write("built")
        return subprocess.CompletedProcess(cmd, 0, "", "")

    monkeypatch.setattr(B.subprocess, "run", run)
    return linked, commands


def test_the_library_is_built_without_torch(stubbed, monkeypatch, capsys):
    linked, commands = stubbed
    monkeypatch.setattr(B.importlib.util, "find_spec", lambda name: None)
    B.build()
    assert linked == ["LIB_PATH", "BENCH_LIB_PATH"] and commands == []
    assert "no ROCm build of torch" in capsys.readouterr().err


def test_the_library_is_built_where_the_extension_cannot_be(stubbed, monkeypatch):
    linked, _ = stubbed
    monkeypatch.setattr(B, "_torch_host_command", lambda out: (["g++", "-o", out], "key"))
    monkeypatch.setattr(B.subprocess, "run", lambda cmd, **kw: subprocess.CompletedProcess(cmd, 1, "", "no such header"))
    with open(B.TORCH_HOST_PATH, "w") as f:
        f.write("an older one")
    with pytest.raises(RuntimeError, match="no such header"):
        B.build()
    assert linked == ["LIB_PATH", "BENCH_LIB_PATH"]
    with open(B.TORCH_HOST_PATH) as f:
        assert f.read() == "an older one"


def test_the_extension_follows_torch(stubbed, monkeypatch):
    _, commands = stubbed
    key = ["torch 1"]
    monkeypatch.setattr(B, "_torch_host_command", lambda out: (["g++", "-o", out], key[0]))
    for want in (1, 1):  # built once, then up to date
        B.build()
        assert len(commands) == want
    key[0] = "torch 2"
    B.build()
    assert len(commands) == 2
    B.build(force=True)
    assert len(commands) == 3
    assert not [f for f in os.listdir(B.OBJ_DIR) if f.startswith("TORCH_HOST_PATH.")]
