"""Face fields of the 4^4 block solver (sap.hip k_sap_reg, rb_push, rb_pull,
k_sap_complete): Schwarz cycles on lattices with two blocks per axis (both
faces of an axis lead to the same block) and with more, both solvers and
boundary conditions, with a twisted mass, several cycles in a row, against
the oracle's FP64 cycles on the same FP32-rounded inputs.  FP32 cycles: 2e-6
of the field's norm for the solution (measured 1.5e-7 per five cycles), 1e-5
for the residual, which is a difference of larger terms; FP16 storage 5e-3
and 1e-2 (2^-11 per stored component and cycle)."""
import ctypes as C

import numpy as np
import pytest

import pyoqh
from helpers import make_oracle

P = C.c_void_p


@pytest.mark.gpu
@pytest.mark.parametrize("L,bc", [((8, 8, 8, 8), 3), ((8, 8, 8, 8), 0), ((16, 8, 24, 8), 3)])
@pytest.mark.parametrize("isolv", [0, 1])
@pytest.mark.parametrize("mu", [0.0, 0.05])
@pytest.mark.parametrize("ncy", [1, 3])
def test_cycles(L, bc, isolv, mu, ncy):
    print("L", L, "bc", bc, "isolv", isolv, "mu", mu, "ncy", ncy, flush=True)
    o, eta, _ = make_oracle(L, None, bc=bc, m0=-0.1, csw=1.77, seed=6)
    eta = eta.astype(np.float32).astype(np.float64)
    lat = pyoqh.Lattice(L, None, bc=bc, m0=-0.1, csw=1.77)
    try:
        V = lat.V
        lat.import_ud(o.ud())
        o.sw_term(3)
        o.set_sap((4, 4, 4, 4), isolv, 4, ncy)
        o.sap_prepare()
        psi, rho = np.zeros((V, 24)), eta.copy()
        for _ in range(ncy):
            o.sap_dble(mu, isolv, 4, psi, rho)
        lib = lat.lib
        lib.sap.argtypes = [C.c_float, C.c_int, C.c_int, P, P]
        bs = np.array((4, 4, 4, 4), np.int32)
        lib.oqh_set_sap_parms(bs.ctypes.data_as(P), isolv, 4, ncy)
        p, r = lat.alloc_s(), lat.alloc_s()
        for prec, tp, tr in ((0, 2e-6, 1e-5), (1, 5e-3, 1e-2)):
            lib.oqh_set_sap_prec(prec)
            lat.put_s(p, np.zeros((V, 24), np.float32))
            lat.put_s(r, eta.astype(np.float32))
            for _ in range(ncy):
                lib.sap(mu, isolv, 4, p, r)
            dp = np.linalg.norm(lat.get_s(p) - psi) / np.linalg.norm(psi)
            dr = np.linalg.norm(lat.get_s(r) - rho) / np.linalg.norm(rho)
            print("precision", prec, "solution", dp, "residual", dr)
            assert dp < tp and dr < tr
    finally:
        lat.lib.oqh_set_sap_prec(0)
        lat.close()
