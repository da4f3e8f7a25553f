"""A tile of a resident 2D launch that waits longer than it may: the launch
ends, the call that waits for it says so, once, and the object goes on with
the per-step kernels.  (The limit is lowered to nothing: the first sample that
is not there at the first look ends the launch.)"""
import numpy as np
import pytest

from geophysics_amd import vti
from test_gpu_run2d_path import Launches, build, models

pytestmark = pytest.mark.gpu
MISSED = "exchange did not arrive"


@pytest.fixture
def wait():
    yield vti.resident_wait
    vti.resident_wait(None)


@pytest.mark.parametrize("form,unsplit,nx,nz", [("gpu", False, 60, 50), ("gpu", True, 700, 301), ("tti", False, 333, 71),
                                                ("gpu", False, 1401, 503)])
def test_steps(wait, form, unsplit, nx, nz):
    with build(form, nx, nz, 20, 80, unsplit) as p:
        p.step(0, 80)
        ref = p.field("P"), p.record()
        p.reset()
        wait(0)
        p.step(0, 80)
        with pytest.raises(vti.VtiError, match=MISSED):
            p.sync()
        wait(None)
        p.sync()
        p.reset()
        with Launches() as n:
            p.step(0, 80)
            assert np.array_equal(p.field("P"), ref[0]) and np.array_equal(p.record(), ref[1])
            assert n() == 0


def test_rtm(wait):
    nx, nz, nt = 333, 71, 40
    with build("gpu", nx, nz, 20, nt, True) as p:
        o = p.rtm_defaults()
        o.nsnap = 3
        obs = np.random.default_rng(3).standard_normal((p.nrec, nt)).astype(np.float32)
        p.rtm_reset()
        p.rtm_shot(o, obs)
        ref = p.rtm_image(finalize=False)
        wait(0)
        with pytest.raises(vti.VtiError, match=MISSED):
            p.rtm_shot(o, obs)
        wait(None)
        p.rtm_reset()
        p.rtm_shot(o, obs)
        got = p.rtm_image(finalize=False)
        assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])


def test_gradient(wait):
    nx, nz, nt = 333, 71, 60
    cfg = vti.cfg_ref2d(vti.MODE_GPU_REF, nx, nz, 10, 10, 20, 1, 20, nt, 1000)
    with vti.Gradient(cfg, fp64=False) as G:
        G.set_model(*models(nx, nz))
        G.set_shot(vti.shot_ref2d(cfg, 1, nx // 2, 0, nz // 2, rec_depth=nz // 2))
        r = np.random.default_rng(1).standard_normal((G.nrec, nt))
        ref = G.run(resid=r, nsnap=3)
        wait(0)
        with pytest.raises(vti.VtiError, match=MISSED):
            G.run(resid=r, nsnap=3)
        wait(None)
        with Launches() as n:
            for _ in range(2):
                got = G.run(resid=r, nsnap=3)
                assert np.array_equal(got["grad_vp"], ref["grad_vp"]) and np.array_equal(got["grad_src"], ref["grad_src"])
            G.forward()
            assert n() == 0
