"""The cell sort in one launch (k_sort_chain) where its items and phases end:
one particle, particle counts around an item of 1024, cell counts around a
scan tile of 4096, more rows of cells than the work map takes in one pass;
with lists rebuilt every step, Verlet lists rebuilt every step by a tiny skin
(the counters must be zero again after each sort) and the default skin.

The bars are those of the parity tests over three steps: trajectories 1e-10,
densities 1e-12."""
import numpy as np
import pytest

from mcf_amd import workloads as W
from mcf_amd.sdpd import SDPD

from gpu_helpers import rel_err, vec_err

pytestmark = pytest.mark.gpu


def box_of(shape, n, seed=7):
    """n particles at random sites of a jittered lattice (dx 1)."""
    dim = len(shape)
    prm = W.tait_box_3d(10, seed=seed).prm.replace(
        num_dim=dim, max_phys=[float(s) for s in shape] + [0.0] * (3 - dim))
    x = W.wrap(W.lattice(dim, list(shape), 1.0, 0.05, seed), prm)
    rng = np.random.default_rng(seed)
    x = x[np.sort(rng.permutation(x.shape[0])[:n])]
    v = rng.normal(0.0, 0.03, size=x.shape)
    return W.Box("sort", prm, x, v, np.full(n, 1.0), np.arange(1, n + 1, dtype=np.int32))


@pytest.mark.parametrize("shape,n", [((10, 10, 10), 1), ((10, 10, 10), 1000), ((40, 40), 1023),
                                     ((40, 40), 1024), ((11, 12, 13), 1025), ((36, 37), 1200),
                                     ((60, 60, 60), 2500), ((400, 400), 4096),
                                     ((20, 130, 130), 5000)])
@pytest.mark.parametrize("skin", [0.0, 1e-9, None])
def test_sort(oracle, shape, n, skin):
    box = box_of(shape, n)
    print(f"sort chain: n={n} {shape} skin={skin}", flush=True)
    with SDPD(box.prm) as g:
        if skin is not None:
            g.set_skin(skin)
        g.upload(box.x, box.v, box.m, box.pid)
        g.integrate_VV(3)
        if skin == 1e-9 and n > 1:
            # (-1: a box too small for a skin rebuilds its lists every step)
            assert g.list_builds() in (4, -1)
        x, v = g.download()
        rho, _ = g.download_density()
        f = g.download_force()
    st = oracle.State(box.prm, box.x, box.v, box.m, box.pid)
    st.prologue(0)
    for k in (1, 2, 3):
        st.vv_step(k)
    assert rel_err(rho, st.rho) < 1e-12
    assert np.abs(x - st.x).max() < 1e-10 * max(shape)
    assert vec_err(v, st.v) < 1e-10
    assert vec_err(f, st.f) < 1e-10


@pytest.mark.parametrize("shape,n", [((17, 16), 255), ((17, 16), 256), ((17, 16), 257),
                                     ((33, 33), 1025), ((64, 64), 4096), ((65, 64), 4097),
                                     ((16, 16, 17), 4096), ((50, 50, 50), 4000),
                                     ((56, 57, 60), 4000)])
@pytest.mark.parametrize("skin", [0.0, 1e-9])
def test_small_sort(oracle, shape, n, skin):
    # k_sort_small where its 256 particles per workgroup, its four particles
    # per thread and its cells in LDS end
    test_sort(oracle, shape, n, skin)
