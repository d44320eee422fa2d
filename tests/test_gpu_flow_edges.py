"""The flow kernel (wflow.hip k_flow) where its storage blocks end inside the
field (V/2 no multiple of 64), with the shortest time extent, and with an odd
and an even number of steps (the gauge field changes place after each):
links within 1e-13 of the oracle after the steps, and the force kept of the
last step within 1e-14 of its scale."""
import numpy as np
import pytest

import pyoqh
import pyoracle as po


@pytest.mark.gpu
@pytest.mark.parametrize("L,T,bc", [((6, 6, 6, 6), None, 3), ((4, 6, 10, 6), None, 0), ((12, 6, 4, 10), (6, 6, 4, 10), 3)])
@pytest.mark.parametrize("n", [1, 2, 5])
def test_flow_ragged(L, T, bc, n):
    print("L", L, "bc", bc, "steps", n, flush=True)
    o = po.Oracle(L, T, bc=bc)
    o.start_ranlux(0, 3)
    o.random_ud()
    lat = pyoqh.Lattice(L, T, bc=bc)
    try:
        lat.import_ud(o.ud())
        lat.lib.fwd_euler(n, 0.02)
        got = lat.export_frc()
        if n > 1:
            o.fwd_euler(n - 1, 0.02)
        ref = o.plaq_frc()
        assert np.abs(got - ref).max() < 1e-14 * np.abs(ref).max()
        o.fwd_euler(1, 0.02)
        assert np.abs(lat.export_ud() - o.ud()).max() < 1e-13
    finally:
        lat.close()
