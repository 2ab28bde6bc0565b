"""The pool of host threads of the transfers (csrc/gcs_host_pool.hpp) where the
system grants none, some or all of its threads: the work is done by those there
are, and no exception reaches the C entry points that use it."""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.mark.parametrize("granted", [0, 1, 3, 64])
def test_pool_does_without_threads_it_is_not_granted(tmp_path, granted):
    exe = tmp_path / "host_pool"
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread",
                    f"-I{os.path.join(ROOT, 'gamera-cube_amd', 'csrc')}",
                    os.path.join(ROOT, "tests", "c", "host_pool.cpp"), "-o", str(exe), "-ldl"],
                   check=True)
    run = subprocess.run([str(exe), str(granted)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout == "ok\n", (run.returncode, run.stdout, run.stderr)
