"""Downloads: the device's reordering (k_to_upload_order) and the pinned pieces
of 1 MiB at the sizes where they end (one particle, a piece to the byte and one
particle more, more pieces than slots).  A sort permutes the particles and
changes none of their values: what comes back equals what was sent, bit for
bit."""
import numpy as np
import pytest

from mcf_amd import workloads as W
from mcf_amd.sdpd import SDPD

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n", [(2, 1), (2, 65536), (2, 65537), (3, 1), (3, 1000), (3, 43690),
                                   (3, 43691), (3, 400000)])
@pytest.mark.parametrize("newtonian", [True, False])
def test_what_was_sent(dim, n, newtonian):
    edge = max(12.0, float(np.ceil(n ** (1 / dim))))
    base = (W.tait_box_3d if newtonian else W.oldroyd_box_3d)(10, seed=3)
    prm = base.prm.replace(num_dim=dim, max_phys=[edge] * dim + [0.0] * (3 - dim))
    rng = np.random.default_rng(n)
    x = rng.random((n, dim)) * edge
    v = rng.normal(0.0, 0.03, size=(n, dim))
    ct = rng.normal(size=(n, dim * dim))
    print(f"download: n={n} dim={dim}", flush=True)
    with SDPD(prm) as g:
        g.upload(x, v, np.full(n, 1.0), np.arange(1, n + 1, dtype=np.int32))
        if not newtonian:
            g.upload_ct(ct)
        for _ in range(2):
            xd, vd = g.download()
            assert np.array_equal(xd, x) and np.array_equal(vd, v)
            if not newtonian:
                assert np.array_equal(g.download_tensors(vgt=False)[0], ct)
            g.build_list()
