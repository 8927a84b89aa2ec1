"""The library's host code on the CPU (tests/host: a runtime that notes the
launches instead of running them): kernels, streams and buffers of a call."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host compiler")
    lib = str(tmp_path_factory.mktemp("host") / "libfake_hip.so")
    subprocess.run([cxx, "-O1", "-std=c++17", "-shared", "-fPIC", "-o", lib, os.path.join(HERE, "fake_hip.cpp")],
                   check=True)
    return lib


@pytest.mark.parametrize("scenario", ["one_run_without_factors", "projections_exist", "general_forms_of_a_face",
                                      "streams_do_not_share_projections", "no_room", "autotuner_times_what_steps_run",
                                      "graphs_of_repeated_calls", "more_waves_than_memory"])
def test_host_path(runtime, scenario):
    r = subprocess.run([sys.executable, os.path.join(HERE, "paths.py"), runtime, scenario], capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
