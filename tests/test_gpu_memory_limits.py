"""Workspaces that only make a call faster when the memory for them is not to be
had: the call goes on without them and gives the same results."""
import ctypes as C

import numpy as np
import pytest

import pyoqh
from helpers import make_oracle

P = C.c_void_p


@pytest.mark.gpu
@pytest.mark.parametrize("L,bc", [((8, 8, 8, 8), 3), ((8, 6, 10, 6), 0)])
def test_flow_in_place(L, bc):
    """Without the second gauge field (576 bytes per point) the flow applies the
    force in place: the same links and force to the last bit."""
    print("L", L, "bc", bc, flush=True)
    out = []
    for limit in (0, 400 * int(np.prod(L))):  # the force takes 256 bytes per point
        lat = pyoqh.Lattice(L, None, bc=bc)
        try:
            lat.lib.start_ranlux(0, 3)
            lat.lib.random_ud()
            lat.lib.oqh_set_alloc_max(limit)
            lat.lib.fwd_euler(3, 0.02)
            lat.lib.oqh_set_alloc_max(0)
            out.append((lat.export_ud(), lat.export_frc()))
        finally:
            lat.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
