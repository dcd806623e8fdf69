"""Small boxes walk their lists with sixteen lanes per particle and build them
with four waves per chunk; larger launches use four lanes and one wave.  Both
visit and add a particle's candidates in list order, so a small box alone and
the same box as the first of a batch that is large enough for the other kernels
must agree bit for bit: rows of 10 to 71 particles (partial groups of 4 and 16),
thinned boxes (particles with no or few neighbours), lists that overflow, every
law with a sixteen-lane walk, and sizes on both sides of the limits."""
import numpy as np
import pytest

from mcf_amd import workloads as W
from mcf_amd.sdpd import SDPD

pytestmark = pytest.mark.gpu

# beyond every limit: 3 * 16384 particles, 1024 chunks
LARGE = 70000


def box_of(shape, law, newtonian, brownian, mixed, drop):
    base = (W.tait_box_3d if newtonian else W.oldroyd_box_3d)(10, seed=7, kt=1e-3)
    dim = len(shape)
    prm = base.prm.replace(num_dim=dim, max_phys=[float(s) for s in shape] + [0.0] * (3 - dim),
                           rhs_force_type=law, Brownian=brownian, precision=1 if mixed else 0)
    x = W.wrap(W.lattice(dim, list(shape), 1.0, 0.05, 7), prm)
    rng = np.random.default_rng(7)
    x = x[rng.random(x.shape[0]) >= drop]
    n = x.shape[0]
    return W.Box("wide", prm, x, rng.normal(0.0, 0.03, size=x.shape), np.full(n, 1.0),
                 np.arange(1, n + 1, dtype=np.int32))


def results(g):
    x, v = g.download()
    return x, v, g.download_density()[0], g.download_force()


def check(box, cap=0, steps=3):
    n = box.n
    k = -(-LARGE // n)
    print(f"wide walk: n={n} x {k} {box.prm.max_phys} law={box.prm.rhs_force_type} "
          f"precision={box.prm.precision} cap={cap}", flush=True)
    with SDPD(box.prm) as g:
        g.set_list_capacity(cap)
        g.upload(box.x, box.v, box.m, box.pid)
        cap = g.list_capacity()
        g.integrate_VV(steps)
        alone = results(g)
    hi = list(box.prm.max_phys[: len(box.prm.max_phys)])
    with SDPD(box.prm) as g:
        g.set_list_capacity(cap)
        g.set_replicas([[0.0] * 3] * k, [hi] * k)
        pid = np.concatenate([box.pid + q * n for q in range(k)]).astype(np.int32)
        g.upload_replicas(np.tile(box.x, (k, 1)), np.tile(box.v, (k, 1)), np.tile(box.m, k), pid,
                          np.repeat(np.arange(k, dtype=np.int32), n))
        g.integrate_VV(steps)
        batch = results(g)
    for a, b in zip(alone, batch):
        assert np.array_equal(a, b[:n])


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("shape,drop", [((10, 12), 0.0), ((71, 13), 0.0), ((10, 10, 10), 0.0),
                                        ((11, 12, 13), 0.6), ((29, 10, 11), 0.97),
                                        ((43, 11, 10), 0.0)])
def test_shapes(shape, drop, mixed):
    check(box_of(shape, 3, True, True, mixed, drop))


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("law,newtonian,brownian", [(3, True, False), (4, True, True),
                                                    (4, True, False), (3, False, True),
                                                    (3, False, False)])
@pytest.mark.parametrize("shape", [(17, 13), (14, 11, 10)])
def test_laws(shape, law, newtonian, brownian, mixed):
    check(box_of(shape, law, newtonian, brownian, mixed, 0.0))


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("cap", [8, 96, 104])
def test_overflow(cap, mixed):
    check(box_of((15, 12, 10), 3, True, True, mixed, 0.05), cap=cap)


@pytest.mark.parametrize("shape", [(25, 25, 26), (26, 25, 26), (33, 33, 28), (37, 37, 35),
                                   (37, 37, 36), (128, 128)])
def test_limits(shape):
    check(box_of(shape, 3, True, True, False, 0.0), steps=2)
