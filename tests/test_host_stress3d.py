"""The kernel that vti_stress3d_name gives is the one the profiles under
profiles/ were taken of, and follows the rules on the grid's size."""
import json
import os

import pytest

from conftest import ROOT
from geophysics_amd import vti


def name(n, unsplit, npml=30):
    return vti.stress3d_name(vti.cfg_ref3d(n, n, n, 10, 10, 10, npml, 1, 20, 10, 1000), unsplit)


@pytest.mark.parametrize("unsplit,profile", [(True, "stress3d_unsplit_traffic.json"), (False, "stress3d_traffic.json")])
def test_profiled_kernels(unsplit, profile):
    with open(os.path.join(ROOT, "profiles", profile)) as f:
        assert name(512, unsplit) == json.load(f)["kernel"]


@pytest.mark.parametrize("n,unsplit,form", [
    (76, False, "4, 0"), (136, False, "4, 1"), (400, False, "4, 1"), (460, False, "16, 1"),
    (124, True, "4, 0"), (152, True, "4, 1"), (198, True, "4, 1"), (204, True, "4, 2"), (240, True, "4, 2"), (600, True, "4, 2")])
def test_rules(n, unsplit, form):
    assert name(n, unsplit) == "vti::s3d::stress3d<%s, %s, false>" % (form, "true" if unsplit else "false")


def test_bad_arguments():
    with pytest.raises(vti.VtiError):
        vti.stress3d_name(vti.cfg_ref2d(vti.MODE_GPU_REF, 60, 50, 10, 10, 20, 1, 20, 10, 1000), True)
