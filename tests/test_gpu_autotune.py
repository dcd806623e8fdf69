"""sdpd_autotune with Verlet lists: it times what a step runs, so the density
shape, which their builds do not take, stays the default whatever was set; the
lists and the trajectory are left as they were.  (Boxes on both sides of 1024
chunk slots, below which builds take four waves per chunk.)"""
import numpy as np
import pytest

from mcf_amd import workloads as W
from mcf_amd.sdpd import SDPD

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side", [12, 45, 64])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("shape", [0, 1, 3])
def test_verlet(side, mixed, shape):
    box = W.tait_box_3d(side, kt=1e-3)
    box = W.mixed(box) if mixed else box
    print(f"autotune: side={side} mixed={mixed} shape={shape}", flush=True)
    with SDPD(box.prm) as a, SDPD(box.prm) as b:
        for g in (a, b):
            g.upload(box.x, box.v, box.m, box.pid)
            g.integrate_VV(1)
        a.set_tuning(shape, 1)
        builds = a.list_builds()
        picked, ms = a.autotune(2)
        assert picked[0] == 0 and picked[1] in (0, 1) and a.tuning() == picked and ms > 0
        assert a.list_builds() == builds
        for g in (a, b):
            g.integrate_VV(2)
        assert np.array_equal(a.download()[0], b.download()[0])
        assert np.array_equal(a.download_force(), b.download_force())
