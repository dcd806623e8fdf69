"""The cell sort of Verlet lists where its kernels' items, phases and sizes end, with
lists that are rebuilt on every step: a skin just above the thinnest that keeps
lists, particles faster than half of it per step.  Each sort finds the counters as
the one before left them, copies the state back and takes new reference positions.

The bars are those of the parity tests over three steps: trajectories 1e-10,
densities 1e-12."""
import numpy as np
import pytest

from mcf_amd import workloads as W
from mcf_amd.sdpd import SDPD

from gpu_helpers import rel_err, vec_err
from test_gpu_sort_chain import box_of

pytestmark = pytest.mark.gpu

SKIN = 4e-6  # 1.3e-6 cut-offs


def fast_box(shape, n):
    box = box_of(shape, n)
    # every particle moves 0.2 * 5e-5 or more per step, five half skins
    box.v[:, 0] = np.where(box.v[:, 0] < 0.0, -0.2, 0.2) + box.v[:, 0]
    return box


def run(box, skin, steps=3):
    with SDPD(box.prm) as g:
        g.set_skin(skin)
        g.upload(box.x, box.v, box.m, box.pid)
        g.integrate_VV(steps)
        if skin > 0.0:
            assert g.list_builds() == steps + 1
        x, v = g.download()
        return x, v, g.download_density()[0], g.download_force()


# k_sort_small (one workgroup, many, its last particles and cells), k_sort_chain
# beyond 4096 particles or 8192 cells
@pytest.mark.parametrize("shape,n", [((17, 16), 1), ((17, 16), 255), ((17, 16), 256),
                                     ((17, 16), 257), ((33, 33), 1025), ((64, 64), 4096),
                                     ((65, 64), 4097), ((16, 16, 17), 4096), ((50, 50, 50), 4000),
                                     ((56, 57, 60), 4000), ((60, 60, 60), 2500), ((400, 400), 4096),
                                     ((20, 130, 130), 5000)])
@pytest.mark.parametrize("mixed", [False, True])
def test_against_oracle(oracle, shape, n, mixed):
    box = fast_box(shape, n)
    print(f"gated sort: n={n} {shape} mixed={mixed}", flush=True)
    x, v, rho, f = run(W.mixed(box) if mixed else box, SKIN)
    st = oracle.State(box.prm, box.x, box.v, box.m, box.pid)
    st.prologue(0)
    for k in (1, 2, 3):
        st.vv_step(k)
    # (mixed precision: the bars of the mixed trajectories)
    assert rel_err(rho, st.rho) < (1e-6 if mixed else 1e-12)
    assert np.abs(x - st.x).max() < (1e-8 if mixed else 1e-10 * max(shape))
    assert vec_err(v, st.v) < (1e-5 if mixed else 1e-10)
    assert vec_err(f, st.f) < (1e-4 if mixed else 1e-10)


# items of 1024 particles on one workgroup each, on fewer than that, beyond 2^20
# particles
@pytest.mark.parametrize("side,n", [(51, 131071), (51, 131072), (51, 131073), (51, 132651),
                                    (102, 1048577)])
def test_items(side, n):
    box = fast_box((side, side, side), n)
    print(f"gated sort: n={n}", flush=True)
    (x, v, rho, f), (x0, v0, rho0, f0) = run(box, SKIN), run(box, 0.0)
    assert rel_err(rho, rho0) < 1e-12
    assert np.abs(x - x0).max() < 1e-10 * side
    assert vec_err(v, v0) < 1e-10
    assert vec_err(f, f0) < 1e-10
