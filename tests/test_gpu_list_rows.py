"""The list build with a wave per chunk (boxes of 1024 chunk slots and more, below
which builds take four waves per chunk) where a stencil row's records end in its
tile of 224: thin boxes, whose rows are mostly empty, to dense ones with rows of
several tiles; boxes that overflow their lists.  Against lists rebuilt every step
by the scan that sums as it goes, in each of its shapes: the same neighbours, so a
density is the same sum of up to a few thousand terms (1e-12; 1e-6 in mixed
precision) and forces agree to 1e-10 of their rms (1e-5)."""
import numpy as np
import pytest

from mcf_amd import workloads as W

from gpu_helpers import rel_err, vec_err
from test_gpu_list_build import evaluate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,edge,per_volume", [(2, 110.0, 12.0), (2, 70.0, 30.0),
                                                 (3, 60.0, 0.01), (3, 45.0, 1.0), (3, 14.0, 24.0)])
@pytest.mark.parametrize("mixed", [False, True])
def test_against_lists_of_every_step(dim, edge, per_volume, mixed):
    n = int(per_volume * edge ** dim)
    prm = W.tait_box_3d(10, seed=5).prm.replace(num_dim=dim,
                                                max_phys=[edge] * dim + [0.0] * (3 - dim))
    rows = (2 * int(edge / (1.0001 * prm.cut_off))) ** (dim - 1)
    assert n // 64 + rows >= 1024
    rng = np.random.default_rng(n)
    x = rng.random((n, dim)) * edge
    x[: n // 4, 0] *= 0.3  # a denser slab
    box = W.Box("rows", prm, x, rng.normal(0.0, 0.03, size=x.shape), np.full(n, 1.0),
                np.arange(1, n + 1, dtype=np.int32))
    print(f"list rows: n={n} dim={dim} mixed={mixed}", flush=True)
    rho0, f0, sig0, _ = evaluate(box, skin=0.0)
    if not mixed:
        for shape in (1, 2, 3):
            rho, f, _, _ = evaluate(box, shape, skin=0.0)
            assert np.array_equal(rho, rho0) and np.array_equal(f, f0)
    for kw in ({}, {"cap": 16}):
        rho, f, sig, builds = evaluate(W.mixed(box) if mixed else box, **kw)
        assert builds == 1
        assert np.array_equal(sig[0], sig0[0]) and np.array_equal(sig[1], sig0[1])
        assert rel_err(rho, rho0) < (1e-6 if mixed else 1e-12)
        assert vec_err(f, f0) < (1e-5 if mixed else 1e-10)
