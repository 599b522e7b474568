"""The build's own rules: the library needs hipcc only, the native host code is an extra, and a library built elsewhere leaves
the tree's own alone. (Nothing is compiled here.)"""
import os
import subprocess
import types

import pytest

from crit_amd import build as builder


class Ran:
    """The commands of a build, run by nobody; `gxx`: what starting the host compiler raises."""
    gxx = None

    def __init__(self):
        self.commands = []

    def run(self, cmd, **_):
        self.commands.append(cmd)
        if cmd[0] == "g++":
            if self.gxx:
                raise self.gxx
            open(cmd[cmd.index("-o") + 1], "w").close()
        return subprocess.CompletedProcess(cmd, 0, "", "")


@pytest.fixture
def ran(monkeypatch, tmp_path):
    found = Ran()
    monkeypatch.setattr(builder, "subprocess", types.SimpleNamespace(run=found.run))
    for name, at in (("LIB", "libcrit_pkv.so"), ("OBJ_DIR", "obj"), ("HOST_LIB", "_pkv_host.so")):
        monkeypatch.setattr(builder, name, str(tmp_path / at))
    monkeypatch.delenv("CRIT_PKV_OUT", raising=False)
    return found


def test_without_a_host_compiler_the_library_is_linked_all_the_same(ran, capsys):
    ran.gxx = FileNotFoundError("g++")
    open(builder.HOST_LIB, "w").close()      # (what an earlier build left: of another ABI, perhaps)
    assert builder.build(verbose=False) == builder.LIB
    assert any(cmd[0] == "hipcc" and builder.LIB in cmd for cmd in ran.commands)
    assert "native host code" in capsys.readouterr().err and not os.path.exists(builder.HOST_LIB)


def test_a_library_built_elsewhere_leaves_the_trees_host_code_alone(ran, monkeypatch, tmp_path):
    monkeypatch.setenv("CRIT_PKV_OUT", str(tmp_path / "other" / "libcrit_pkv.so"))
    assert builder.build(verbose=False) == os.environ["CRIT_PKV_OUT"]
    assert not any(cmd[0] == "g++" for cmd in ran.commands) and not os.path.exists(builder.HOST_LIB)


def test_the_host_code_arrives_whole_or_not_at_all(ran):
    builder.build(verbose=False)
    made = next(cmd for cmd in ran.commands if cmd[0] == "g++")
    assert made[made.index("-o") + 1] != builder.HOST_LIB
    assert sorted(os.listdir(os.path.dirname(builder.HOST_LIB))) == ["_pkv_host.so", "obj"]
