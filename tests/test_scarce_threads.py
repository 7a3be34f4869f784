"""Large results without the helper threads: page faults ahead and the copy out of
the staging buffers go on with as many threads as can be made (tests/cpp/
scarce_threads.cpp makes pthread_create and operator new fail)."""
import os
import subprocess

import pytest

from conftest import ROOT

LIBDIR = os.path.join(ROOT, "parallel-task1_amd", "lib")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = tmp_path_factory.mktemp("scarce") / "scarce_threads"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-rdynamic", "-pthread",
                    os.path.join(ROOT, "tests", "cpp", "scarce_threads.cpp"), "-L" + LIBDIR,
                    "-lsssp_mi355x", "-ldl", "-Wl,-rpath," + LIBDIR, "-o", str(out)],
                   check=True, capture_output=True, text=True)
    return str(out)


def test_prefault_without_threads_or_memory(program):
    r = subprocess.run([program, "pages"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "pages ok" in r.stdout, r.stdout + r.stderr


@pytest.mark.gpu
def test_large_results_without_threads(gpu, program):
    r = subprocess.run([program, "gpu"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "gpu ok" in r.stdout, r.stdout + r.stderr
