"""The in-tree build recompiles what a change reaches, and nothing else."""
import importlib.util
import os

import pytest

from conftest import PKG


@pytest.fixture
def build(monkeypatch, tmp_path):
    """build.py on a tree of its own, with a compiler that writes its output's name."""
    spec = importlib.util.spec_from_file_location("wm_build_under_test", os.path.join(PKG, "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    csrc, include = tmp_path / "pkg" / "csrc", tmp_path / "include"
    csrc.mkdir(parents=True), include.mkdir()
    (include / "api.h").write_text("")
    (csrc / "common.hpp").write_text('#include "deep.hpp"\n')
    (csrc / "deep.hpp").write_text("")
    (csrc / "kernel.hip").write_text('#include <vector>\n#include "common.hpp"\n')
    (csrc / "kernel_wide.hip").write_text('#define WIDE 1\n#include "kernel.hip"\n')
    (csrc / "other.hip").write_text('  # include "../../include/api.h"\n')
    made = []

    class Compiler:
        returncode = 0

        def __init__(self, cmd, **_):
            made.append(os.path.basename(cmd[cmd.index("-o") + 1]))
            with open(cmd[cmd.index("-o") + 1], "w"):
                pass

        def communicate(self):
            return "", None

    monkeypatch.setattr(mod.subprocess, "Popen", Compiler)
    monkeypatch.setattr(mod, "_run", Compiler)
    monkeypatch.setattr(mod, "__file__", str(tmp_path / "build.py"))
    (tmp_path / "build.py").write_text("")
    for name, value in (("CSRC", csrc), ("INCLUDE", include), ("HIP_LIB", tmp_path / "pkg" / "library.so")):
        monkeypatch.setattr(mod, name, str(value))

    def rebuilt(changed=None):
        """What is made again after `changed`, with every other file an hour old."""
        for root, _, files in os.walk(tmp_path):
            for f in files:
                os.utime(os.path.join(root, f), (1e9, 1e9))
        if changed:
            os.utime(tmp_path / changed, (1e9 + 60, 1e9 + 60))
        made.clear()
        mod.build_hip_library()
        return set(made)

    mod.build_hip_library()
    return rebuilt


@pytest.mark.parametrize("changed,objects", [
    (None, set()),
    ("pkg/csrc/kernel.hip", {"kernel.o", "kernel_wide.o"}),  # a wrapper's object holds the source that it includes
    ("pkg/csrc/kernel_wide.hip", {"kernel_wide.o"}),
    ("pkg/csrc/deep.hpp", {"kernel.o", "kernel_wide.o"}),
    ("include/api.h", {"other.o"}),
    ("build.py", {"kernel.o", "kernel_wide.o", "other.o"}),  # flags
])
def test_objects_that_a_change_reaches(build, changed, objects):
    assert build(changed) == (objects | {"library.so"} if objects else set())
