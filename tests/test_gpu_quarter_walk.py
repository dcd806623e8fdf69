"""The walk of Verlet lists with four lanes per particle (k_density_walk,
k_force_walk) at the sizes where its 16-particle quarters and batches end:
rows of 15 to 130 particles (chunks of 64 cut into partial quarters), one
quarter or a whole chunk per workgroup, particles without any neighbour,
pairs across every face in both image conventions, every force law.

The bars are those of the parity tests: FP64 densities 1e-13 and forces 1e-12
per evaluation; here two steps are taken so that the density comes from the
walk too, whose trajectories agree to 1e-10 (densities 1e-12), and mixed
precision to 1e-5 of FP64 forces."""
import numpy as np
import pytest

from mcf_amd import workloads as W
from mcf_amd.sdpd import SDPD

from gpu_helpers import rel_err, vec_err

pytestmark = pytest.mark.gpu


def box_of(shape, law=3, newtonian=True, brownian=True, symmetry=True, seed=3, drop=0.0):
    """A jittered lattice box of the given edges (dx 1), thinned at random."""
    base = (W.tait_box_3d if newtonian else W.oldroyd_box_3d)(10, seed=seed)
    dim = len(shape)
    prm = base.prm.replace(num_dim=dim, max_phys=[float(s) for s in shape] + [0.0] * (3 - dim),
                           rhs_force_type=law, Brownian=brownian, symmetry=symmetry)
    x = W.wrap(W.lattice(dim, list(shape), 1.0, 0.05, seed), prm)
    rng = np.random.default_rng(seed)
    x = x[rng.random(x.shape[0]) >= drop]
    # the x faces lie on a lattice plane: pairs across them from the start
    x[:, 0] = np.where(x[:, 0] < 0.5, 0.0, x[:, 0])
    v = rng.normal(0.0, 0.03, size=x.shape)
    n = x.shape[0]
    return W.Box("quarter", prm, x, v, np.full(n, 1.0), np.arange(1, n + 1, dtype=np.int32))


def run(box, steps=2):
    with SDPD(box.prm) as g:
        g.upload(box.x, box.v, box.m, box.pid)
        g.integrate_VV(steps)
        x, v = g.download()
        rho, _ = g.download_density()
        return x, v, rho, g.download_force()


SHAPES = [(10, 12), (11, 13), (43, 10), (44, 10), (87, 11), (10, 10, 10), (14, 11, 10),
          (29, 10, 11), (58, 10, 10)]


def check(oracle, box):
    print(f"quarter walk: n={box.n} law={box.prm.rhs_force_type} {box.prm.max_phys}", flush=True)
    x, v, rho, f = run(box)
    st = oracle.State(box.prm, box.x, box.v, box.m, box.pid)
    st.prologue(0)
    st.vv_step(1)
    st.vv_step(2)
    assert rel_err(rho, st.rho) < 1e-12
    assert vec_err(v, st.v) < 1e-10
    assert vec_err(f, st.f) < 1e-10


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("symmetry", [True, False])
def test_row_lengths(oracle, shape, symmetry):
    check(oracle, box_of(shape, symmetry=symmetry))


@pytest.mark.parametrize("law,newtonian,brownian",
                         [(1, True, False), (2, True, True), (4, True, True), (3, True, False),
                          (2, False, True), (3, False, True), (4, False, False)])
def test_force_laws(oracle, law, newtonian, brownian):
    check(oracle, box_of((15, 10, 11), law, newtonian, brownian))


@pytest.mark.parametrize("drop", [0.5, 0.9, 0.995])
def test_sparse(oracle, drop):
    check(oracle, box_of((31, 12, 10), brownian=True, drop=drop))


def test_whole_chunks_and_mixed():
    # enough chunks that a workgroup takes all four quarters of one
    box = W.tait_box_3d(64, kt=1e-3)
    print(f"quarter walk: n={box.n}", flush=True)
    x, v, rho, f = run(box)
    xm, vm, rhom, fm = run(W.mixed(box))
    assert rel_err(rhom, rho) < 1e-6
    assert vec_err(fm, f) < 1e-5
    # the rescans of overflowed lists sum one particle per lane: the same bits
    with SDPD(box.prm) as g:
        g.set_list_capacity(48)
        g.upload(box.x, box.v, box.m, box.pid)
        g.integrate_VV(2)
        assert np.array_equal(g.download_density()[0], rho)
        assert np.array_equal(g.download_force(), f)
