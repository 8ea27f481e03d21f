"""the build takes torch's paths from the interpreter that runs it, not from the python3 on PATH"""
import sys

from blockwise_int8_linear_amd import build


def test_make_is_given_the_running_interpreter(monkeypatch):
    commands = []

    class Done:
        returncode, stdout = 0, ""
    monkeypatch.setattr(build.subprocess, "run", lambda cmd, **kw: commands.append(cmd) or Done())
    build.build()
    assert f"PYTHON={sys.executable}" in commands[0]
