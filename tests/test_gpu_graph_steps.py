"""sdpd_step's graphs of four steps: calls whose steps hold none, one, several of
them and every remainder, on either parity of the sort's buffers (lists rebuilt
every step swap them) and after eager work in between, equal direct launches bit
for bit."""
import numpy as np
import pytest

from mcf_amd import workloads as W
from mcf_amd.sdpd import SDPD

pytestmark = pytest.mark.gpu

BOXES = {
    "tait": lambda: W.tait_box_3d(12, kt=1e-3),
    "tait_mixed": lambda: W.mixed(W.tait_box_3d(17, kt=1e-3)),
    "oldroyd": lambda: W.oldroyd_box_3d(11),
    "wave": lambda: W.shear_wave_2d(32),
}


@pytest.mark.parametrize("name", list(BOXES))
@pytest.mark.parametrize("skin", [-1.0, 0.0])
def test_replays_equal_direct_launches(name, skin):
    box = BOXES[name]()
    print(f"graph steps: {name} skin={skin}", flush=True)
    with SDPD(box.prm) as a, SDPD(box.prm) as b:
        b.set_graphs(False)
        for g in (a, b):
            g.set_skin(skin)
            g.upload(box.x, box.v, box.m, box.pid)
        for chunk in (9, 13, 6, 1, 5, 8, 12):
            for g in (a, b):
                g.integrate_VV(chunk)
            for u, w in zip(a.download(), b.download()):
                assert np.array_equal(u, w), chunk
            assert np.array_equal(a.download_force(), b.download_force()), chunk
            assert a.step == b.step and a.list_builds() == b.list_builds()
            if chunk in (6, 5):
                for g in (a, b):
                    g.evaluate()
