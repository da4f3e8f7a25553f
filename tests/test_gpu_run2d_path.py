"""Which path a call takes: launches of the resident 2D kernel, counted, for
the calls that are meant to use it and for those that keep the per-step
kernels.  (tests/test_gpu_run2d.py compares the results of the two; without
the count it would pass if neither side ran the resident kernel.)"""
import threading

import numpy as np
import pytest

from geophysics_amd import vti

pytestmark = pytest.mark.gpu


class Launches:
    """with Launches() as n: ...; n() is the launches so far"""

    def __enter__(self):
        self.n0 = vti.resident_launches()
        return lambda: vti.resident_launches() - self.n0

    def __exit__(self, *exc):
        return False


def models(nx, nz, seed=1):
    rng = np.random.default_rng(seed)
    vp = (2200.0 + 600.0 * rng.random((nx, nz))).astype(np.float32)
    ep = (0.2 * rng.random((nx, nz))).astype(np.float32)
    return vp, ep, (0.5 * ep).astype(np.float32)


def build(form, nx, nz, npml, nt, unsplit=False):
    mode = {"cpu": vti.MODE_CPU_REF, "omp": vti.MODE_OMP_REF}.get(form, vti.MODE_GPU_REF)
    cfg = vti.cfg_ref2d(mode, nx, nz, 10, 10, npml, 1, 20, nt, 1000)
    p = vti.Propagator(cfg, *models(nx, nz))
    if form == "tti":
        p.set_theta(np.full((nx, nz), 10.0, dtype=np.float32), degrees=True)
    p.set_unsplit(unsplit)
    p.set_shot(vti.shot_ref2d(cfg, 1, nx // 2, 0, nz // 2, rec_depth=max(1, nz // 3)))
    p.reset()
    return p


# one tile; the smallest tiles; one to eight rows a thread (TTI: to six)
@pytest.mark.parametrize("form,unsplit,nx,nz,npml", [
    ("gpu", False, 16, 17, 0), ("gpu", True, 11, 13, 5), ("cpu", False, 60, 50, 20), ("gpu", False, 333, 71, 20),
    ("gpu", True, 64, 403, 9), ("gpu", False, 1401, 503, 20), ("gpu", True, 2001, 602, 30),
    ("gpu", False, 2401, 803, 20), ("tti", False, 15, 12, 4), ("tti", False, 700, 301, 20),
    ("tti", False, 1401, 503, 20), ("tti", False, 2300, 440, 20)])
def test_steps_are_resident(form, unsplit, nx, nz, npml):
    with build(form, nx, nz, npml, 120, unsplit) as p, Launches() as n:
        p.step(0, 40)
        assert n() == 1
        p.step(40, 8)
        assert n() == 2
        p.step(48, 7)             # too few steps
        assert n() == 2
        p.run()
        assert n() == 3
        p.prof_enable(True)       # timed launch by launch
        p.step(0, 40)
        assert n() == 3


def test_short_runs_of_a_fresh_context_keep_the_per_step_kernels():
    """The plan and its memory pay from 24 steps on, in whatever calls."""
    for calls, launches in (((23,), 0), ((24,), 1), ((8, 15), 0), ((8, 3, 13), 1), ((16, 8, 8), 2), ((23, 7, 8), 1)):
        with build("gpu", 120, 90, 20, 40) as p, Launches() as n:
            it = 0
            for k in calls:
                p.step(it, k)
                it += k
            assert n() == launches, calls


# too large for the chip, and the form whose sums are in double
@pytest.mark.parametrize("form,nx,nz,npml", [("gpu", 2500, 1000, 20), ("tti", 2401, 803, 20), ("omp", 120, 90, 0)])
def test_steps_keep_the_per_step_kernels(form, nx, nz, npml):
    with build(form, nx, nz, npml, 40) as p, Launches() as n:
        p.step(0, 40)
        p.sync()
        assert n() == 0


# a shot is two launches: the first sweep and the rest
@pytest.mark.parametrize("nx,nz,npml,nt,nsnap,per_shot", [
    (16, 17, 4, 8, 0, 2), (15, 12, 4, 40, 2, 2), (64, 403, 9, 33, 4, 2), (1401, 503, 20, 20, 2, 2),
    (1901, 602, 20, 16, 2, 2), (2401, 1003, 20, 10, 2, 0), (60, 50, 3, 40, 4, 0), (60, 50, 20, 7, 2, 0)])
def test_rtm_shots(nx, nz, npml, nt, nsnap, per_shot):
    obs = np.random.default_rng(3).standard_normal((nx, nt)).astype(np.float32)
    with build("gpu", nx, nz, npml, nt, True) as p, Launches() as n:
        o = p.rtm_defaults()
        o.nsnap = nsnap
        o.inject_z = npml + nz // 2 - 2
        for k in (1, 2):
            p.rtm_shot(o, obs[:p.nrec])
            assert n() == k * per_shot
        p.adcig_config(2)         # gathers go step by step
        p.rtm_shot(o, obs[:p.nrec])
        assert n() == 2 * per_shot


@pytest.mark.parametrize("large,resident", [((2401, 403), True), ((2401, 1003), False)])
def test_batches(large, resident):
    sizes, nt = [(900, 301), (333, 71), (1200, 500), (16, 17), (60, 50), large, (700, 301)], 12
    cfgs = [vti.cfg_ref2d(vti.MODE_GPU_REF, nx, nz, 10, 10, 4 + k, k % 2, 20, nt, 1000)
            for k, (nx, nz) in enumerate(sizes)]
    shots = [vti.shot_ref2d(c, 1, nx // 2, 0, 3) for c, (nx, nz) in zip(cfgs, sizes)]
    obs = [np.ones((s.rec_nx, nt), dtype=np.float32) for s in shots]
    o = vti.rtm_defaults(2)
    o.nsnap = 2
    with vti.Batch(cfgs, shots, [models(*s) for s in sizes]) as B, Launches() as n:
        B.rtm(o, obs)
        first = n()
        # several parts, two launches each
        assert first >= 4 and first % 2 == 0 if resident else first == 0
        B.rtm(o, obs)
        assert n() == 2 * first


@pytest.mark.parametrize("nx,nz,npml,fp64,resident", [(16, 17, 4, False, True), (333, 71, 20, False, True),
                                                      (700, 301, 20, False, True), (333, 71, 20, True, False),
                                                      (2401, 1003, 20, False, False)])
def test_gradients(nx, nz, npml, fp64, resident):
    nt = 40
    cfg = vti.cfg_ref2d(vti.MODE_GPU_REF, nx, nz, 10, 10, npml, 1, 20, nt, 1000)
    with vti.Gradient(cfg, fp64=fp64) as G, Launches() as n:
        G.set_model(*models(nx, nz))
        G.set_shot(vti.shot_ref2d(cfg, 1, nx // 2, 0, nz // 2, rec_depth=nz // 2))
        for k in (1, 2):
            G.forward()
            G.run(resid=np.ones((G.nrec, nt)), nsnap=3)
            assert n() == (2 * k if resident else 0)   # the modelled record; the first sweep


@pytest.mark.parametrize("nt,launches", [(12, (0, 0, 0)), (24, (0, 1, 2)), (40, (1, 2, 3))])
def test_short_gradients(nt, launches):
    """A few steps pay from the second sweep of an object on, or not at all."""
    nx, nz = 120, 90
    cfg = vti.cfg_ref2d(vti.MODE_GPU_REF, nx, nz, 10, 10, 20, 1, 20, nt, 1000)
    with vti.Gradient(cfg, fp64=False) as G, Launches() as n:
        G.set_model(*models(nx, nz))
        G.set_shot(vti.shot_ref2d(cfg, 1, nx // 2, 0, nz // 2, rec_depth=nz // 2))
        out = []
        for k in launches:
            out.append(G.forward())
            assert n() == k
        assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


def test_threads_of_one_launch_shape():
    """Four threads whose grids share a launch shape (threads and rows a strip)
    and need different amounts of LDS: every call is a resident launch, and the
    fields are those of each context alone."""
    sizes = [(1400, 503), (1300, 503), (1150, 503), (1400, 503)]
    alone, got, count = {}, {}, {}

    def work(k, into):
        nx, nz = sizes[k]
        with build("gpu", nx, nz, 20, 64) as p, Launches() as n:
            for _ in range(20):
                p.step(0, 64)
            into[k] = p.field("P")
            count[k] = n()

    for k in range(len(sizes)):
        work(k, alone)
        assert count[k] == 20
    count.clear()
    th = [threading.Thread(target=work, args=(k, got)) for k in range(len(sizes))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert count == {k: 20 for k in range(len(sizes))}
    for k in alone:
        assert np.array_equal(alone[k], got[k]), k
