"""The downloads' reordering against numpy, and an upload index out of range: it
writes nothing and reports, and the download then fails."""
import ctypes as C

import numpy as np
import pytest

from mcf_amd.sdpd import load_library

from hip_buffers import DeviceArray, synchronize

pytestmark = pytest.mark.gpu

# sdpd::launch_to_upload_order(hipStream_t, int, int, const int32_t*, const double*, double*, int32_t*)
SYMBOL = "_ZN4sdpd22launch_to_upload_orderEP12ihipStream_tiiPKiPKdPdPi"


@pytest.mark.parametrize("n", [1, 255, 257])
@pytest.mark.parametrize("comps", [1, 9])
@pytest.mark.parametrize("wrong", [None, -1, "n", 2 ** 31 - 1])
def test_upload_order(n, comps, wrong):
    launch = getattr(load_library(), SYMBOL)
    launch.restype = None
    launch.argtypes = [C.c_void_p, C.c_int, C.c_int] + [C.c_void_p] * 4
    rng = np.random.default_rng(n)
    perm = rng.permutation(n).astype(np.int32)
    src = rng.normal(size=(comps, n))
    want = np.full((n, comps), -7.0)
    want[perm] = src.T
    if wrong is not None:
        want[perm[n // 2]] = -7.0
        perm[n // 2] = n if wrong == "n" else wrong
    print(f"upload order: n={n} comps={comps} wrong={wrong}", flush=True)
    p, s, d, flag = (DeviceArray(a) for a in (perm, src, np.full((n, comps), -7.0),
                                              np.zeros(1, np.int32)))
    launch(None, n, comps, p.addr, s.addr, d.addr, flag.addr)
    synchronize()
    assert np.array_equal(d.get(), want)
    assert flag.get()[0] == (wrong is not None)
