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


CALLS = {
    # these wait for the stream
    "sync": lambda p, d: p.sync(), "get_record": lambda p, d: p.record(), "get_field": lambda p, d: p.field("P"),
    "set_field": lambda p, d: p.set_field("u", np.zeros(p.shape, dtype=np.float32)),
    "set_stream": lambda p, d: vti.check(vti.lib().vti_set_stream(p.h, None)),
    "prof_enable": lambda p, d: p.prof_enable(False), "prof_read": lambda p, d: p.prof_read(),
    "adcig_get": lambda p, d: p.adcig(),
    # these queue work on the state or the record
    "step": lambda p, d: p.step(0, 2), "update_vel": lambda p, d: p.update_vel(0),
    "update_stress": lambda p, d: p.update_stress(0), "mute": lambda p, d: p.mute(60, 0, 2, 1),
    "save_state": lambda p, d: vti.check(vti.lib().vti_save_state(p.h, d.data_ptr())),
    "image_accumulate": lambda p, d: vti.check(vti.lib().vti_image_accumulate(p.h, p.h, d.data_ptr(), None, 0)),
    "adcig_accumulate": lambda p, d: vti.check(vti.lib().vti_adcig_accumulate(p.h, p.h)),
}


@pytest.mark.parametrize("call", CALLS)
def test_every_call_reports(wait, call):
    import torch
    with build("gpu", 120, 90, 20, 80) as p:
        d = torch.zeros(p.state_bytes() // 4, device="cuda")
        torch.cuda.synchronize()
        p.adcig_config(2)
        p.step(0, 80)
        CALLS[call](p, d)
        wait(0)
        p.step(0, 80)
        torch.cuda.synchronize()        # the device, without a call on the context
        with pytest.raises(vti.VtiError, match=MISSED):
            CALLS[call](p, d)
        p.sync()                        # once
        p.reset()
        CALLS[call](p, d)
        p.sync()


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
