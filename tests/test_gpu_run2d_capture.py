"""The first resident 2D steps of a context while another stream is being
captured into a graph (torch's default, global capture mode, which forbids
allocations and waits in all threads): they run, and the capture is unharmed."""
import threading

import numpy as np
import pytest

from geophysics_amd import vti
from test_gpu_run2d_path import Launches, build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["gpu", "tti after gpu"])
@pytest.mark.parametrize("thread", [False, True])
def test_first_steps_beside_a_capture(form, thread):
    import torch

    def make():
        p = build("gpu", 120, 90, 20, 80)
        if form != "gpu":
            p.step(0, 40)
            p.set_theta(np.full((120, 90), 10.0, dtype=np.float32), degrees=True)
            p.reset()
        p.sync()
        return p

    with make() as a, make() as b:
        a.step(0, 80)
        ref = a.field("P"), a.record()
        x = torch.zeros(1000, device="cuda")
        g = torch.cuda.CUDAGraph()
        n = []

        def steps():
            with Launches() as count:
                b.step(0, 80)
                n.append(count())

        with torch.cuda.graph(g):
            x.add_(1.0)
            if thread:
                t = threading.Thread(target=steps)
                t.start()
                t.join()
            else:
                steps()
        assert n == [1]
        assert np.array_equal(b.field("P"), ref[0]) and np.array_equal(b.record(), ref[1])
        for k in range(3):
            g.replay()
            torch.cuda.synchronize()
            assert float(x.min()) == float(x.max()) == k + 1
            b.reset()
            b.step(0, 80)
            assert np.array_equal(b.record(), ref[1])
