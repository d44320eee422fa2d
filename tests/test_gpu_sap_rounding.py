"""Rounding error of the FP32 Schwarz cycles (sap.hip) against the FP64 cycles on
the device: five cycles of four MinRes steps, relative error of the solution
and of the residual in the 2-norm.  The bounds are what kernels that round
every product and every sum separately (k_sap_blocks on these inputs, on 4^4
blocks an earlier k_sap_reg with the hops summed from zero) leave: blocks in
registers or on the chip must not be less precise.  The numbers are sums over
2 10^5 to 1.6 10^6 components, so they hardly depend on the fields."""
import ctypes as C

import numpy as np
import pytest

import pyoqh

P = C.c_void_p


@pytest.mark.gpu
@pytest.mark.parametrize("bs,L,T,isolv,sol,res", [
    ((4, 4, 4, 4), (16, 16, 16, 16), (8, 8, 8, 8), 0, 1.352e-7, 3.852e-7),
    ((4, 4, 4, 4), (16, 16, 16, 16), (8, 8, 8, 8), 1, 1.410e-7, 3.761e-7),
    ((8, 8, 8, 8), (16, 16, 16, 16), (8, 8, 8, 8), 0, 1.163e-7, 3.603e-7),
    ((8, 8, 8, 8), (16, 16, 16, 16), (8, 8, 8, 8), 1, 1.205e-7, 3.353e-7),
    ((8, 4, 4, 4), (16, 8, 8, 8), (8, 8, 8, 8), 0, 1.184e-7, 3.530e-7),
    ((8, 4, 4, 4), (16, 8, 8, 8), (8, 8, 8, 8), 1, 1.220e-7, 3.425e-7),
    ((6, 6, 6, 6), (12, 12, 12, 12), None, 0, 1.171e-7, 3.476e-7),
    ((6, 6, 6, 6), (12, 12, 12, 12), None, 1, 1.213e-7, 3.340e-7)])
def test_rounding(bs, L, T, isolv, sol, res):
    print("blocks", bs, "L", L, "isolv", isolv, flush=True)
    lat = pyoqh.Lattice(L, T, bc=3, m0=-0.1, csw=1.77)
    try:
        lib, V = lat.lib, lat.V
        lib.start_ranlux(0, 6)
        lib.random_ud()
        lib.set_ud_phase()
        assert lat.sw_term(3) == 0
        lib.sap.argtypes = [C.c_float, C.c_int, C.c_int, P, P]
        lib.oqh_set_sap_parms((C.c_int * 4)(*bs), isolv, 4, 5)
        eta = np.random.default_rng(6).standard_normal((V, 24)).astype(np.float32)
        p, r = lat.alloc_s(), lat.alloc_s()
        out = []
        for prec in (2, 0):
            lib.oqh_set_sap_prec(prec)
            lat.put_s(p, np.zeros((V, 24), np.float32))
            lat.put_s(r, eta)
            for _ in range(5):
                lib.sap(0.05, isolv, 4, p, r)
            out.append((lat.get_s(p).astype(np.float64), lat.get_s(r).astype(np.float64)))
        d = [np.linalg.norm(a - b) / np.linalg.norm(b) for a, b in zip(out[1], out[0])]
        print("solution", d[0], "residual", d[1])
        assert d[0] <= sol and d[1] <= res
    finally:
        lat.lib.oqh_set_sap_prec(0)
        lat.close()
