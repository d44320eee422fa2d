"""Copies between host arrays and the device at the edges of the chunked path
(state.hip host_copy): just below and above its least size of 16 MiB, last
chunks that are not full, fewer and more chunks than threads, an array that
does not start on a page, memory that the caller has pinned.  Bytes are
unchanged, outside the range too."""
import ctypes as C

import numpy as np
import pytest
import torch

import pyoqh


@pytest.fixture(scope="module")
def lat():
    lat = pyoqh.Lattice((24, 24, 24, 24), bc=3, m0=0.1, csw=1.0)
    yield lat
    lat.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [87381, 87382, 109227, 174763, 331776])  # sites of 192 bytes
@pytest.mark.parametrize("pinned", [False, True])
def test_round_trip(lat, n, pinned):
    print("sites", n, "pinned", pinned, flush=True)
    rng = np.random.default_rng(n)
    src = rng.random((n, 24))
    pad = 3  # doubles before the array
    if pinned:
        buf = torch.empty(n * 24 + 2 * pad, dtype=torch.float64, pin_memory=True).numpy()
    else:
        buf = np.empty(n * 24 + 2 * pad)
    buf[:] = -1.0
    host = buf[pad:pad + n * 24]
    host[:] = src.reshape(-1)
    f = lat.alloc_sd()
    lat.lib.oqh_import_sd(f, host.ctypes.data, n)
    host[:] = 0.0  # free to change on return
    assert np.array_equal(lat.get_sd(f, n), src)
    lat.lib.oqh_export_sd(f, host.ctypes.data, n)
    assert np.array_equal(host, src.reshape(-1))
    assert (buf[:pad] == -1.0).all() and (buf[-pad:] == -1.0).all()
    lat.free(f)


@pytest.mark.gpu
def test_links(lat):
    ud = np.random.default_rng(1).random((4 * lat.V, 18))
    lat.import_ud(ud)
    assert np.array_equal(lat.export_ud(), ud)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1000, 331776])
@pytest.mark.parametrize("pinned", [False, True])
def test_argument_free_on_return(lat, n, pinned):
    """A host array given to an operation on a device field may be changed as soon
    as the call returns, also if work queued before keeps the device busy."""
    print("sites", n, "pinned", pinned, flush=True)
    src = np.random.default_rng(n).random((n, 24))
    if pinned:
        host = torch.empty(n * 24, dtype=torch.float64, pin_memory=True).numpy()
    else:
        host = np.empty(n * 24)
    host[:] = src.reshape(-1)
    lat.lib.assign_sd2s.argtypes = [C.c_int, C.c_int, C.c_void_p, C.c_void_p]
    lat.lib.start_ranlux(0, 1)
    lat.lib.random_ud()
    lat.sw_term(3)
    f, s, r = lat.alloc_s(), lat.alloc_sd(), lat.alloc_sd()
    lat.lib.assign_sd2s(n, 0, host.ctypes.data, f)
    lat.sync()
    for _ in range(100):  # 12 ms
        lat.lib.Dw_dble(0.0, s, r)
    lat.lib.assign_sd2s(n, 0, host.ctypes.data, f)
    host[:] = 0.0
    assert np.array_equal(lat.get_s(f, n), src.astype(np.float32))
    for p in (f, s, r):
        lat.free(p)
