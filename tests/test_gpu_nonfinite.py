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


@pytest.mark.parametrize("mixed", [False, True])
def test_position(mixed):
    # A particle without neighbours, whose lists hold particles in the skin,
    # moves to a position that is not a number: the others go on as without it.
    # (Fixed-point units are 3e-9 and the velocities of the records 6e-8 of
    # theirs: 1e-6 for densities, 1e-5 for forces; a neighbour adds 1e-3.)
    box = W.tait_box_3d(12, kt=1e-3)
    i = box.n - 1
    box.x[i] = 11.3
    r = distances(box.x, i, box.prm)
    keep = (r > 1.001 * box.prm.cut_off) | (np.arange(box.n) == i)
    assert (r[keep] < box.prm.cut_off + 0.8).sum() > 10
    prm = W.mixed(box).prm if mixed else box.prm
    x, v, m, pid = box.x[keep], box.v[keep], box.m[keep], box.pid[keep]
    out = []
    for vi in (0.0, np.nan):
        v[-1] = vi
        with SDPD(prm) as g:
            g.set_skin(0.9)
            g.upload(x, v, m, pid)
            g.integrate_VV(3)
            out.append((g.download()[0], g.download_density()[0], g.download_force()))
            builds = g.list_builds()
    (x0, rho0, f0), (x1, rho1, f1) = out
    assert np.isnan(x1[-1]).all()
    assert np.abs(x1[:-1] - x0[:-1]).max() < 1e-8
    assert np.abs(rho1[:-1] / rho0[:-1] - 1.0).max() < 1e-6
    assert np.abs(f1[:-1] - f0[:-1]).max() < 1e-5 * np.abs(f0).max()
    # the lists are rebuilt once, without it
    assert builds == (2 if mixed else 1)


@pytest.mark.parametrize("lists", ["verlet", "every step", "mixed"])
@pytest.mark.parametrize("speed", [np.nan, np.inf, 1e9, 1e300])
def test_lost_between_sheared_faces(lists, speed):
    # A particle that leaves the box, or whose position is not a number, has no
    # window in the sheared frame: its cell's is taken, and the particles beyond
    # its neighbours' neighbours go on.
    box = W.tait_box_3d(20, kt=1e-3)
    prm = box.prm.replace(le_dim=2, le_v_lower=[-0.3, 0, 0], le_v_upper=[0.3, 0, 0])
    i = int(np.argmin(np.abs(box.x - 10.0).sum(1)))
    far = distances(box.x, i, prm) > 3.2 * prm.cut_off
    assert far.sum() > 1000
    box.v[i] = speed
    print(f"lost between sheared faces: {lists} speed={speed}", flush=True)
    with SDPD(prm.replace(precision=1) if lists == "mixed" else prm) as g:
        if lists == "every step":
            g.set_skin(0.0)
        g.upload(box.x, box.v, box.m, box.pid)
        g.integrate_VV(2)
        x, v = g.download()
        rho = g.download_density()[0]
    assert np.isfinite(x[far]).all() and np.isfinite(v[far]).all()
    assert (np.abs(rho[far] - 1.0) < 0.2).all()
