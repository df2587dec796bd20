"""The field copies between host and device without a GPU: their source is
compiled for the CPU against a model of the few runtime calls that it makes
(hostcopy_host.cpp)."""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("hostcopy") / "hostcopy")
    src = os.path.join(ROOT, "energy-stability_amd", "csrc")
    subprocess.run(["g++", "-std=c++20", "-O2", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + src,
                    os.path.join(ROOT, "tests", "hostcopy_host.cpp"), "-o", exe, "-lpthread"], check=True)
    return exe


@pytest.mark.parametrize("what", ["trips", "device", "pinned", "signals", "threads"])
def test_copies(program, what):
    """trips: what comes back is what was set, over every way a copy goes; device: from a thread whose current
    device is not the context's; pinned: a buffer that the runtime knows is copied in one piece;
    signals: the helper threads block them; threads: all of them are joined once the last context is closed."""
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr
