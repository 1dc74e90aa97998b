"""What the build asks for, without running a compiler."""
import importlib.util
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_the_library_is_built_without_torch(monkeypatch):
    """A user of the C ABI alone needs hipcc and no torch: only the host extension is left out."""
    spec = importlib.util.spec_from_file_location("standalone_build", os.path.join(ROOT, "bitladder_amd", "build.py"))
    B = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(B)
    commands = []

    class Done:
        returncode, stdout = 0, ""

        def __init__(self, cmd, **kw):
            commands.append(cmd)

        def communicate(self):
            return "", None

    monkeypatch.setattr(subprocess, "Popen", Done)
    monkeypatch.setattr(subprocess, "run", lambda cmd, **kw: Done(cmd))

    def outputs():
        commands.clear()
        B.build()
        return {os.path.basename(cmd[cmd.index("-o") + 1]) for cmd in commands}

    everything = outputs()
    assert "_hostpath.so" in everything
    monkeypatch.setitem(sys.modules, "torch", None)
    assert outputs() == everything - {"_hostpath.so"}
