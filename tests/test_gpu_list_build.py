"""The list build of Verlet lists (list_scan) where a stencil row's records end
in its tile: thin to dense boxes, whose rows hold from none to more records
than a tile of 128 or 224 takes, each density shape, boxes that overflow their
lists.  Against lists rebuilt every step by the scan that sums as it goes: the
same neighbours, so a density is the same sum of up to 1000 terms (1e-12) and
forces agree to 1e-10 of the largest."""
import numpy as np
import pytest

from mcf_amd import workloads as W
from mcf_amd.sdpd import SDPD

from gpu_helpers import rel_err, vec_err

pytestmark = pytest.mark.gpu


def evaluate(box, shape=0, **kw):
    with SDPD(box.prm) as g:
        if "skin" in kw:
            g.set_skin(kw["skin"])
        if "cap" in kw:
            g.set_list_capacity(kw["cap"])
        g.upload(box.x, box.v, box.m, box.pid)
        g.set_tuning(shape, 1)
        g.evaluate()
        return g.download_density()[0], g.download_force(), g.neighbor_signature(), g.list_builds()


@pytest.mark.parametrize("dim,per_volume", [(2, 0.02), (2, 1.0), (2, 12.0), (3, 0.01), (3, 1.0),
                                            (3, 8.0)])
@pytest.mark.parametrize("shape", [0, 1, 3])
def test_against_lists_of_every_step(dim, per_volume, shape):
    edge = 40.0 if dim == 2 else 14.0
    n = int(per_volume * edge ** dim)
    prm = W.tait_box_3d(10, seed=5).prm.replace(num_dim=dim,
                                                max_phys=[edge] * dim + [0.0] * (3 - dim))
    rng = np.random.default_rng(n)
    x = rng.random((n, dim)) * edge
    x[: n // 4, 0] *= 0.3  # a denser slab
    box = W.Box("lists", prm, x, rng.normal(0.0, 0.03, size=x.shape), np.full(n, 1.0),
                np.arange(1, n + 1, dtype=np.int32))
    print(f"list build: n={n} dim={dim} shape={shape}", flush=True)
    rho0, f0, sig0, builds0 = evaluate(box, skin=0.0)
    assert builds0 == -1
    for kw in ({}, {"cap": 16}):
        rho, f, sig, builds = evaluate(box, shape, **kw)
        assert builds == 1
        assert np.array_equal(sig[0], sig0[0]) and np.array_equal(sig[1], sig0[1])
        assert rel_err(rho, rho0) < 1e-12
        assert vec_err(f, f0) < 1e-10
