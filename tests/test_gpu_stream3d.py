"""3D steps on grids on both sides of the sizes at which the velocity and the
stress update change the fields that bypass the caches, in 4-plane chunks
with a remainder: bit for bit the oracle's."""
import numpy as np
import pytest

from geophysics_amd import vti
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


# fields of 10, 27, 36, 68 and 120 MB: all cached; (split) model and split
# fields streamed; u, v, w too; (unsplit) P and Q too
@pytest.mark.parametrize("nx,ny,nz,unsplit", [(90, 101, 95, 0), (90, 101, 95, 1), (150, 133, 130, 0), (150, 133, 130, 1),
                                              (170, 169, 170, 1), (217, 218, 190, 0), (217, 218, 190, 1), (262, 263, 270, 1)])
def test_3d_steps_match_oracle_at_every_cache_rule(nx, ny, nz, unsplit):
    npml, nt = 20, 5
    rng = np.random.default_rng(nx + unsplit)
    vp = (2200.0 + 600.0 * rng.random((ny, nx, nz), dtype=np.float32)).astype(np.float32)
    e = 0.2 * rng.random((ny, nx, nz), dtype=np.float32)
    d = (0.5 * e).astype(np.float32)
    cfg = vti.cfg_ref3d(nx, ny, nz, 10, 10, 10, npml, 1, 25, nt, 800)
    with vti.Propagator(cfg, vp, e, d) as prop:
        prop.set_unsplit(bool(unsplit))
        prop.set_shot(vti.shot_ref3d(cfg, 0, nx // 2, 0, ny // 2, 0, 4, 0, rec_depth=3, rec_step=2))
        prop.run()
        rec = prop.record()
        f = {k: prop.field(k) for k in ("u", "v", "w", "P", "Q")}
    p = po.params_gpu3d(nx, ny, nz, 10, 10, 10, npml, 1, 25, 0, nx // 2, 0, ny // 2, 0, 4, 0, nt, 800, 3, 2)
    p.unsplit = unsplit
    sim = po.Sim(p, vp, e, d, "f32")
    ref = sim.run()
    assert np.abs(ref).max() > 0
    assert np.array_equal(rec, ref)
    for k, v in f.items():
        assert np.array_equal(v, sim.field(k)), k
