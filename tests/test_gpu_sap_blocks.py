"""Schwarz cycles with blocks other than 4^4: the kernel that keeps the block's
spinors on the chip (sap.hip k_sap_lds; each of its three work-group sizes,
with idle lanes), the one that shares a block among work-groups
(k_sap_cluster, 2, 4, 8 and 16 of them) and the one for other large blocks, both
solvers and boundary conditions, with a twisted mass, against the oracle's FP64 cycles on
the same FP32-rounded inputs: 2e-6 of the field's norm for the solution and
1e-5 for the residual (measured 1.5e-7 and 3e-7 after five cycles)."""
import ctypes as C

import numpy as np
import pytest

import pyoqh
from helpers import make_oracle

P = C.c_void_p


@pytest.mark.gpu
@pytest.mark.parametrize("bs,L,T", [((8, 4, 4, 4), (16, 8, 8, 8), None), ((4, 4, 6, 4), (8, 8, 12, 8), (8, 8, 6, 8)), ((6, 4, 4, 4), (12, 8, 8, 8), (6, 8, 8, 8)),
                                    ((4, 6, 6, 6), (8, 12, 12, 12), (8, 6, 6, 6)),
                                    ((8, 8, 4, 4), (16, 16, 8, 8), (8, 8, 8, 8)), ((6, 6, 6, 6), (12, 12, 12, 12), None),
                                    ((4, 8, 6, 8), (8, 16, 12, 16), (8, 8, 6, 8)),
                                    ((8, 8, 8, 4), (16, 16, 16, 8), (8, 8, 8, 8)), ((8, 8, 8, 8), (16, 16, 16, 16), (8, 8, 8, 8))])
@pytest.mark.parametrize("isolv", [0, 1])
@pytest.mark.parametrize("bc,mu", [(3, 0.0), (0, 0.05)])
def test_cycles(bs, L, T, isolv, bc, mu):
    print("blocks", bs, "L", L, "bc", bc, "isolv", isolv, "mu", mu, flush=True)
    ncy = 2
    o, eta, _ = make_oracle(L, T, bc=bc, m0=-0.1, csw=1.77, seed=6)
    eta = eta.astype(np.float32).astype(np.float64)
    lat = pyoqh.Lattice(L, T, bc=bc, m0=-0.1, csw=1.77)
    try:
        V = lat.V
        lat.import_ud(o.ud())
        o.sw_term(3)
        o.set_sap(bs, isolv, 3, ncy)
        o.sap_prepare()
        psi, rho = np.zeros((V, 24)), eta.copy()
        for _ in range(ncy):
            o.sap_dble(mu, isolv, 3, psi, rho)
        lib = lat.lib
        lib.sap.argtypes = [C.c_float, C.c_int, C.c_int, P, P]
        b = np.array(bs, np.int32)
        lib.oqh_set_sap_parms(b.ctypes.data_as(P), isolv, 3, ncy)
        p, r = lat.alloc_s(), lat.alloc_s()
        lat.put_s(r, eta.astype(np.float32))
        for _ in range(ncy):
            lib.sap(mu, isolv, 3, p, r)
        dp = np.linalg.norm(lat.get_s(p) - psi) / np.linalg.norm(psi)
        dr = np.linalg.norm(lat.get_s(r) - rho) / np.linalg.norm(rho)
        print("solution", dp, "residual", dr)
        assert dp < 2e-6 and dr < 1e-5
    finally:
        lat.close()
