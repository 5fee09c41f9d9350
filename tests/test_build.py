"""A library appears whole under its name: processes that find it missing and build it together never load a part of one."""
import os
import subprocess

import pytest

from nuvec_amd import build


def test_a_library_appears_whole(tmp_path, monkeypatch):
    target = str(tmp_path / "_native.so")
    monkeypatch.setattr(build, "NATIVE", target)
    outputs = []

    def compiler(cmd, **kwargs):
        out = cmd[cmd.index("-o") + 1]
        outputs.append(out)
        with open(out, "w") as f:
            f.write("half")
            f.flush()
            assert not os.path.exists(target) or open(target).read() == "whole"
            f.seek(0)
            f.write("whole")
        return subprocess.CompletedProcess(cmd, 1 if len(outputs) == 3 else 0, "", "no")
    monkeypatch.setattr(build.subprocess, "run", compiler)
    for _ in range(2):
        assert build.build_native() == target and open(target).read() == "whole"
    with pytest.raises(RuntimeError, match="native.cpp"):
        build.build_native()
    assert open(target).read() == "whole" and os.listdir(tmp_path) == ["_native.so"]  # (a build that fails leaves nothing behind)
