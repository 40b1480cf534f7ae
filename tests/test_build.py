"""The build's steps, with the compilers stood in for: the library needs neither PyTorch nor g++, and a failure names its tool."""
import os

import pytest

from tritonbench_amd import build


@pytest.mark.parametrize("jobs", [0, 1])
def test_the_library_is_in_place_when_the_binding_fails(monkeypatch, tmp_path, jobs):
    monkeypatch.setattr(build, "LIB_DIR", str(tmp_path))
    monkeypatch.setattr(build, "LIB_PATH", str(tmp_path / "lib.so"))
    monkeypatch.setattr(build, "BINDING_PATH", str(tmp_path / "binding.so"))
    monkeypatch.setattr(build, "BUILD_DIR", str(tmp_path / "obj"))
    monkeypatch.setattr(build, "find_hipcc", lambda: "hipcc")

    def run(cmd, verbose):
        if cmd[0] == "g++":
            raise RuntimeError("no g++ here")
        open(cmd[cmd.index("-o") + 1], "w").close()
    monkeypatch.setattr(build, "_run", run)
    with pytest.raises(RuntimeError, match="no g\\+\\+ here"):
        build.build_library(jobs=jobs)
    assert os.path.exists(build.LIB_PATH) and not os.path.exists(build.BINDING_PATH)


def test_a_failure_names_the_tool():
    with pytest.raises(RuntimeError, match="^false failed"):
        build._run(["/bin/false"], False)
