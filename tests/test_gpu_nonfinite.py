"""A particle whose values are not finite reaches the particles inside its
cut-off and no others: what lies between the cut-off and the skin of a Verlet
list is left out, as the reference leaves it out (pp_interaction.inc:37-46).
Every other particle keeps the bits it has without it."""
import numpy as np
import pytest

from mcf_amd import workloads as W
from mcf_amd.sdpd import SDPD

pytestmark = pytest.mark.gpu


def largest_skin(prm):
    edge = min(prm.length[: prm.num_dim])
    return 2.0 * edge / (2 * int(edge / (1.0001 * prm.cut_off))) - prm.cut_off


def distances(x, i, prm):
    d = x - x[i]
    L = np.array(prm.length[: prm.num_dim])
    return np.sqrt(((d - L * np.rint(d / L)) ** 2).sum(1))


def evaluate(box, cap):
    with SDPD(box.prm) as g:
        g.set_skin(0.9 * largest_skin(box.prm))
        if cap:
            g.set_list_capacity(cap)
        g.upload(box.x, box.v, box.m, box.pid)
        g.evaluate()
        out = [g.download_force()]
        if not box.prm.Newtonian:
            out.append(g.download_tensors()[1])
        return out


def check(box, cap=0):
    # a particle at the middle of the box, so that all of its lists hold it
    i = int(np.argmin(np.abs(box.x - 0.5 * np.array(box.prm.length[: box.prm.num_dim])).sum(1)))
    r, rc = distances(box.x, i, box.prm), box.prm.cut_off
    inside = r < rc
    ring = (r > 1.0001 * rc) & (r < rc + 0.9 * largest_skin(box.prm))
    assert ring.any() and inside.sum() > 4
    want = evaluate(box, cap)
    box.v[i] = np.nan
    for a, b in zip(evaluate(box, cap), want):
        assert np.array_equal(a[~inside], b[~inside])
        assert not np.isfinite(a[inside]).all(1).any()


# the walks: sixteen lanes with the rescan, sixteen without, four
@pytest.mark.parametrize("shape", [(12, 12, 12), (20, 20), (26, 26, 26), (37, 37, 37)])
@pytest.mark.parametrize("newtonian,law", [(True, 1), (True, 2), (True, 3), (True, 4), (False, 2),
                                           (False, 3), (False, 4)])
@pytest.mark.parametrize("mixed", [False, True])
def test_velocity(shape, newtonian, law, mixed):
    dim = len(shape)
    prm = (W.tait_box_3d if newtonian else W.oldroyd_box_3d)(10).prm.replace(
        num_dim=dim, max_phys=[float(s) for s in shape] + [0.0] * (3 - dim), rhs_force_type=law,
        Brownian=law in (2, 3) or (newtonian and law == 4))
    x = W.wrap(W.lattice(dim, list(shape), 1.0, 0.05, 3), prm)
    n = x.shape[0]
    v = np.random.default_rng(4).normal(0.0, 0.03, size=x.shape)
    print(f"not finite: n={n} dim={dim} newtonian={newtonian} law={law} mixed={mixed}", flush=True)
    box = W.Box("nan", prm, x, v, np.full(n, 1.0), np.arange(1, n + 1, dtype=np.int32))
    check(W.mixed(box) if mixed else box)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("side", [12, 26])
def test_velocity_overflowed_lists(mixed, side):
    # every chunk is scanned again
    box = W.tait_box_3d(side, kt=1e-3)
    print(f"not finite, overflowed lists: side={side} mixed={mixed}", flush=True)
    check(W.mixed(box) if mixed else box, cap=8)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("brownian", [False, True])
def test_velocity_lucy_and_quiet(mixed, brownian):
    box = W.tait_box_3d(14, kt=1e-3, brownian=brownian)
    for kernel in (1, 2):
        b = W.tait_box_3d(14, kt=1e-3, brownian=brownian)
        b.prm = box.prm.replace(kernel_type=kernel)
        print(f"not finite: kernel={kernel} brownian={brownian} mixed={mixed}", flush=True)
        check(W.mixed(b) if mixed else b)


def test_velocity_between_sheared_faces():
    box = W.tait_box_3d(16, kt=1e-3)
    box.prm = box.prm.replace(le_dim=2, le_v_lower=[-0.3, 0, 0], le_v_upper=[0.3, 0, 0])
    print("not finite: sheared faces", flush=True)
    check(box)
