"""particles_compute_pressure by itself: the pressures and the factors of the pair
forces are those that the density pass has stored, so the forces keep their
bits, with every force law, where the number density is far from 1."""
import numpy as np
import pytest

from mcf_amd import workloads as W

from gpu_helpers import gpu_evaluate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("newtonian,law", [(True, 1), (True, 2), (True, 3), (True, 4), (False, 2),
                                           (False, 3), (False, 4)])
@pytest.mark.parametrize("mixed", [False, True])
def test_forces_after_the_pressure(newtonian, law, mixed):
    box = W.shear_wave_2d(64, brownian=law in (2, 3))
    box.prm = box.prm.replace(rhs_force_type=law, Newtonian=newtonian, tau=0.1, n_p=1.0, kt_p=0.5)
    print(f"pressure: newtonian={newtonian} law={law} mixed={mixed}", flush=True)
    g = gpu_evaluate(W.mixed(box) if mixed else box, step=3)
    rho, p = g.download_density()
    f = g.download_force()
    g.compute_pressure()
    g.compute_interaction()
    assert np.array_equal(g.download_density()[1], p)
    assert np.array_equal(g.download_force(), f)
    g.close()
