"""A resident 2D launch that is refused, at any point of a call: the call goes
on with the per-step kernels and gives what it gives without the refusal, bit
for bit (the two kinds of kernel do the same arithmetic)."""
import numpy as np
import pytest

from geophysics_amd import vti
from test_gpu_run2d_path import Launches, build, models

pytestmark = pytest.mark.gpu


@pytest.fixture
def limit():
    yield vti.resident_limit
    vti.resident_limit(None)


def test_steps(limit):
    out = []
    for n in (None, 1, 0):
        with build("gpu", 333, 71, 20, 40) as p:
            limit(n)
            p.step(0, 26)
            p.step(26, 14)
            out.append((p.field("P"), p.field("pz"), p.record()))
    for o in out[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(o, out[0]))


# one checkpoint that steps start from, several, all states kept; whole and
# packed (unsplit) checkpoints; images and records of a first shot kept
@pytest.mark.parametrize("nx,nz,npml,nt,nsnap", [(15, 12, 4, 40, 1), (333, 71, 20, 70, 3), (64, 403, 9, 33, 0)])
@pytest.mark.parametrize("unsplit,illum_mode", [(False, 0), (True, 1)])
def test_rtm(limit, unsplit, illum_mode, nx, nz, npml, nt, nsnap):
    out = []
    for n in (None, 3, 2, 1, 0):      # two launches a shot
        with build("gpu", nx, nz, npml, nt, unsplit) as p, Launches() as count:
            o = p.rtm_defaults()
            o.nsnap, o.illum_mode = nsnap, illum_mode
            o.inject_z = npml + nz // 2 - 2
            obs = np.random.default_rng(3).standard_normal((p.nrec, nt)).astype(np.float32)
            limit(n)
            steps = [p.rtm_shot(o, obs) for _ in range(2)]
            assert count() == (4 if n is None else n)
            img, ill = p.rtm_image(finalize=False)
            out.append((img, ill, p.record()) + tuple(p.field(k) for k in ("u", "w", "P", "Q", "px", "qz")) + (steps,))
    assert np.abs(out[0][0]).max() > 0
    for o in out[1:]:
        assert o[-1] == out[0][-1]
        for k, (a, b) in enumerate(zip(o[:-1], out[0][:-1])):
            if unsplit and k >= 7:      # no split fields in the unsplit interior
                continue
            assert np.array_equal(a, b), k


@pytest.mark.parametrize("unsplit", [False, True])
def test_batch(limit, unsplit):
    sizes, nt = [(900, 301), (333, 71), (1200, 500), (16, 17), (60, 50), (700, 301)], 16
    cfgs = [vti.cfg_ref2d(vti.MODE_GPU_REF, nx, nz, 10, 10, 4 + k, k % 2, 20, nt, 1000)
            for k, (nx, nz) in enumerate(sizes)]
    shots = [vti.shot_ref2d(c, 1, nx // 2, 0, 3) for c, (nx, nz) in zip(cfgs, sizes)]
    rng = np.random.default_rng(5)
    obs = [rng.standard_normal((s.rec_nx, nt)).astype(np.float32) for s in shots]
    o = vti.rtm_defaults(2)
    o.nsnap = 3
    with vti.Batch(cfgs, shots, [models(*s) for s in sizes]) as B:
        B.set_unsplit(unsplit)

        def shot():
            steps = B.rtm(o, obs)
            return steps, [B.image(k) for k in range(len(sizes))], [B.record(k) for k in range(len(sizes))]

        with Launches() as count:
            ref = shot()
            launches = count()
        assert launches >= 4             # at least two parts, so that a refusal can fall between two
        for n in range(launches):
            limit(n)
            with Launches() as count:
                got = shot()
                assert count() == n
            assert got[0] == ref[0]
            for k in range(len(sizes)):
                assert np.abs(ref[1][k][0]).max() > 0
                assert np.array_equal(got[1][k][0], ref[1][k][0]) and np.array_equal(got[1][k][1], ref[1][k][1]), (n, k)
                assert np.array_equal(got[2][k], ref[2][k]), (n, k)


def test_gradient(limit):
    nx, nz, nt = 333, 71, 60
    cfg = vti.cfg_ref2d(vti.MODE_GPU_REF, nx, nz, 10, 10, 20, 1, 20, nt, 1000)
    with vti.Gradient(cfg, fp64=False) as G, Launches() as count:
        G.set_model(*models(nx, nz))
        G.set_shot(vti.shot_ref2d(cfg, 1, nx // 2, 0, nz // 2, rec_depth=nz // 2))
        r = np.random.default_rng(1).standard_normal((G.nrec, nt))
        ref, rec = G.run(resid=r, nsnap=3), G.forward()
        assert count() == 2
        limit(0)                         # after launches that went well
        got, rec0 = G.run(resid=r, nsnap=3), G.forward()
        assert count() == 2
        limit(None)
        again = G.run(resid=r, nsnap=3)
        assert count() == 3              # the object is resident again
        assert np.array_equal(rec0, rec)
        for k in ("grad_vp", "grad_src"):
            assert np.array_equal(got[k], ref[k]) and np.array_equal(again[k], ref[k]), k
