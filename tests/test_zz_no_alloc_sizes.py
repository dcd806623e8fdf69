"""sdpd_evaluate_noalloc beyond the boxes that one workgroup's LDS sorts (4096
particles, 8192 cells) and next to its limit, against the context path: the same
sums in the same order, bit for bit, in calls that alternate between sizes and
precisions, so that each finds another's leftovers in the static array."""
import numpy as np
import pytest

from mcf_amd import workloads as W
from mcf_amd.sdpd import SDPDError

from test_gpu_sort_chain import box_of
from test_zz_no_alloc import announce, context_path, noalloc

pytestmark = pytest.mark.gpu


def thin(edge, n=1000):
    return box_of((edge, edge, edge), n)


BOXES = [
    lambda: W.tait_box_3d(17, kt=1e-3),
    lambda: W.mixed(W.tait_box_3d(39, kt=1e-3)),
    lambda: W.tait_box_3d(32, kt=1e-3),
    lambda: W.mixed(W.tait_box_3d(17, kt=1e-3)),
    lambda: W.shear_wave_2d(250),
    lambda: thin(63),
    lambda: W.mixed(W.shear_wave_2d(250)),
    lambda: W.tait_box_3d(39, kt=1e-3),
    lambda: W.mixed(thin(63)),
    lambda: W.mixed(W.tait_box_3d(32, kt=1e-3)),
    lambda: W.tait_box_3d(12, kt=1e-3),
]


def test_sizes():
    for k, make in enumerate(BOXES):
        box = make()
        announce(f"noalloc sizes: {box.name} n={box.n}")
        for a, b in zip(noalloc(box, 3 + k), context_path(box, 3 + k)):
            assert np.array_equal(a, b)


def asked(n, nm, mixed):
    """Bytes by which a 3D box of (2 nm)^3 sort cells is refused: its buffers with
    lists of 8 entries in blocks of whole chunks, each on 256 bytes (the array held
    32 MiB and these before it grew for longer lists)."""
    cells, rows = (2 * nm) ** 3, (2 * nm) ** 2
    chunks = (n + 63) // 64 + rows
    sizes = ([24 * n] * 4 + [8 * n] * 2 + [4 * n] * 6          # x, v, m, pid, perm, rep, copies
             + [24 * n] + [8 * n] * 4 + [4 * n] * 2            # f, rho, p, factors, key, slot
             + [4 * cells, 4 * (cells + 1)] + [4 * n] * 2      # count, start, unsorted, key_sorted
             + [16 * n] + ([16 * n] * 2 if mixed else [64 * n])  # positions, records
             + [256] + [4 * rows] * 3 + [8, 32]                # geometry, step, times
             + [4 * rows, 4 * (rows + 1), 4 * chunks, 4 * ((max(cells, rows) + 4095) // 4096 + 1)]
             + [4 * n] * 3                                     # counts
             + [8 * 64 * 4 * ((chunks + 7) // 8 * 8)]          # lists
             + [16, 8, 24 * n])                                # gate, displacement, reference
    return sum(-(-s // 256) * 256 for s in sizes)


@pytest.mark.parametrize("mixed", [False, True])
def test_limit(mixed):
    n = 1000
    nm = max(k for k in range(3, 200) if asked(n, k, mixed) <= 32 << 20)
    for k, held in ((nm, True), (nm + 1, False)):
        edge = 3.01 * k
        prm = W.tait_box_3d(10).prm.replace(max_phys=[edge] * 3)
        rng = np.random.default_rng(k)
        x = np.minimum(rng.random((n, 3)) * edge, np.nextafter(edge, 0.0))
        x[: n // 2] *= 0.02  # some have neighbours
        box = W.Box("limit", prm, x, rng.normal(0.0, 0.03, (n, 3)), np.full(n, 1.0),
                    np.arange(1, n + 1, dtype=np.int32))
        box = W.mixed(box) if mixed else box
        announce(f"noalloc limit: {k} cells of PPM's grid per edge, held={held}")
        if not held:
            with pytest.raises(SDPDError):
                noalloc(box, 1)
            continue
        for a, b in zip(noalloc(box, 1), context_path(box, 1)):
            assert np.array_equal(a, b)
