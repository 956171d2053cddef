"""The engine's host logic (memory, admission, chunks) against a stand-in for the
HIP runtime whose device is host memory: engine_host.cpp, linked to the built
library.  No GPU and no kernel is involved."""
import os
import subprocess

import pytest

from suli_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("engine_host") / "engine_host")
    lib = os.path.dirname(build.LIB)
    r = subprocess.run([build.hipcc(), "-std=c++17", "-O1", "-Wall", "-Wno-unused-result",
                        os.path.join(HERE, "engine_host.cpp"),
                        "-o", exe, "-L", lib, "-l:" + os.path.basename(build.LIB), f"-Wl,-rpath,{lib}"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


@pytest.mark.parametrize("scenario", ["fallback", "cached", "failed_setup", "beside", "batch", "chunk", "masks"])
def test_scenario(program, scenario):
    r = subprocess.run([program, scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
