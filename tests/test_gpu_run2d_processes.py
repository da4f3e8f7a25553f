"""Processes that share the device: the runtime refuses some of their resident
2D launches while another process has its own, at any point of an RTM's
schedule.  Every call of each gives what the per-step kernels give."""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu


def work():
    from geophysics_amd import vti
    vti.resident_wait(5000000)
    rng = np.random.default_rng(1)
    nx, nz, nt = 333, 181, 60
    cfg = vti.cfg_ref2d(vti.MODE_GPU_REF, nx, nz, 10, 10, 20, 1, 20, nt, 1000)
    vp = (2200.0 + 600.0 * rng.random((nx, nz))).astype(np.float32)
    ep = (0.2 * rng.random((nx, nz))).astype(np.float32)
    shot = vti.shot_ref2d(cfg, 1, nx // 2, 0, nz // 2, rec_depth=3)
    with vti.Propagator(cfg, vp, ep, ep) as p, vti.Gradient(cfg, fp64=False) as G:
        p.set_unsplit(True)
        p.set_shot(shot)
        G.set_model(vp, ep, ep)
        G.set_shot(shot)
        o = p.rtm_defaults()
        o.nsnap = 4
        obs = rng.standard_normal((p.nrec, nt)).astype(np.float32)
        resid = rng.standard_normal((G.nrec, nt))

        def all_of_it():
            p.run()
            rec = p.record()
            p.rtm_reset()
            p.rtm_shot(o, obs)
            return (rec,) + p.rtm_image(finalize=False) + (G.run(resid=resid, nsnap=4)["grad_vp"],)

        vti.resident_limit(0)
        ref = all_of_it()
        vti.resident_limit(None)
        for k in range(40):
            for a, b in zip(all_of_it(), ref):
                assert np.array_equal(a, b), k
    print("equal, %d resident launches" % vti.resident_launches())


def test_three_processes():
    code = "import sys; sys.path[:0] = [%r, %r]; import test_gpu_run2d_processes as t; t.work()" % (
        ROOT, os.path.join(ROOT, "tests"))
    run = [subprocess.Popen([sys.executable, "-c", code], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
           for _ in range(3)]
    out = [r.communicate(timeout=100)[0] for r in run]
    print("\n".join(out), flush=True)
    assert all(r.returncode == 0 and "equal" in o for r, o in zip(run, out)), out
