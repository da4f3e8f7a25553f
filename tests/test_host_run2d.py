"""Host side of the resident 2D steps without a device: tests/host_run2d.hip
over a made-up runtime, one scenario a test."""
import os
import subprocess

import pytest

from conftest import ROOT
from geophysics_amd import build

SCENARIOS = ["lds_attribute", "refused_step", "launch_order", "short_calls", "shared_device", "refused_program", "missed_exchange",
             "plans"]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("host_run2d")
    obj, exe = str(d / "host_run2d.o"), str(d / "host_run2d")
    # host pass only; without a unique id the device code's symbol has one name
    flags = [f for f in build.FLAGS if f != "-shared"] + ["--cuda-host-only", "-fuse-cuid=none"]
    subprocess.run([build.HIPCC] + flags + ["-c", os.path.join(ROOT, "tests", "host_run2d.hip"), "-o", obj], check=True)
    subprocess.run(["g++", obj, "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("scenario", SCENARIOS)
def test_scenario(program, scenario):
    r = subprocess.run([program, scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
