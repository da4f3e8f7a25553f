"""3D split steps on a grid of more than 500 MB a field, where the stress update
marches chunks of 16 planes instead of 4 (469 updated planes: 29 chunks and 5
planes), bit for bit the fused kernel's, which has one chunk length for all
sizes and is compared with the oracle elsewhere."""
import numpy as np
import pytest

from geophysics_amd import vti

pytestmark = pytest.mark.gpu

def test_largest_split_chunks_equal_the_fused_step():
    import torch
    nx, ny, nz, npml, nt = 480, 437, 470, 20, 3
    rng = np.random.default_rng(4)
    ep = rng.random((ny, nx, nz), dtype=np.float32)
    vp = 2200.0 + 600.0 * ep
    ep *= 0.2
    cfg = vti.cfg_ref3d(nx, ny, nz, 10, 10, 10, npml, 1, 25, nt, 800)
    shot = vti.shot_ref3d(cfg, 0, nx // 2, 0, ny // 2, 0, 4, 0, rec_depth=3, rec_step=2)
    torch.manual_seed(1)
    out = []
    for fused in (False, True):
        with vti.Propagator(cfg, vp, ep, ep) as p:
            n = p.state_bytes() // 4
            assert n == 11 * 477 * 520 * 512 and 4e-6 * (n // 11) > 500.0
            if not out:
                start = torch.randn(n, device="cuda")       # every cell of every field
                torch.cuda.synchronize()
            p.set_fused(fused)
            p.set_shot(shot)
            p.reset()
            p.load_state(start.data_ptr())
            p.step(0, nt)
            end = torch.empty(n, device="cuda")
            torch.cuda.synchronize()
            p.save_state(end.data_ptr())
            out.append((end, p.record()))
    (a, ra), (b, rb) = out
    assert np.isfinite(ra).all() and np.abs(ra).max() > 0 and np.array_equal(ra, rb)
    for k in range(11):
        x, y, z = (t[k * (n // 11):(k + 1) * (n // 11)] for t in (a, b, start))
        assert bool(torch.isfinite(x).all()) and not torch.equal(x, z), k
        assert torch.equal(x, y), k
