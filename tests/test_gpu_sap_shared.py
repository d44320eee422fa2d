"""Schwarz blocks shared by several work-groups (sap.hip k_sap_cluster) where
the other tests do not go: more work-groups in a launch than the chip holds (2048
of 8^4 blocks at 32^4, at most 512 at once), 32 and 64 work-groups per block, and
the even-odd twisted mass (eoflg).  Two cycles, both solvers, against the
FP64 cycles of k_sap_blocks on the device on the same FP32 inputs, within 2e-6 of
the field's norm for the solution and 1e-5 for the residual, the bounds of
the smaller lattices, whose FP64 cycles are compared with the oracle."""
import ctypes as C

import numpy as np
import pytest

import pyoqh

P = C.c_void_p


@pytest.mark.gpu
@pytest.mark.parametrize("bs,L,T", [((8, 8, 8, 8), (32, 32, 32, 32), (8, 8, 8, 8)),
                                    ((16, 8, 8, 8), (32, 16, 16, 16), (8, 8, 8, 8)),
                                    ((16, 16, 8, 8), (32, 32, 16, 16), (8, 8, 8, 8))])
@pytest.mark.parametrize("isolv", [0, 1])
@pytest.mark.parametrize("bc,eoflg", [(3, 1), (0, 0)])
def test_cycles(bs, L, T, isolv, bc, eoflg):
    print("blocks", bs, "L", L, "bc", bc, "isolv", isolv, "eoflg", eoflg, flush=True)
    lat = pyoqh.Lattice(L, T, bc=bc, m0=-0.1, csw=1.77, eoflg=eoflg)
    try:
        lib, V = lat.lib, lat.V
        lib.start_ranlux(0, 6)
        lib.random_ud()
        assert lat.sw_term(3) == 0
        lib.sap.argtypes = [C.c_float, C.c_int, C.c_int, P, P]
        lib.oqh_set_sap_parms((C.c_int * 4)(*bs), isolv, 4, 2)
        rng = np.random.default_rng(6)
        e, p, r = lat.alloc_s(), lat.alloc_s(), lat.alloc_s()
        lat.put_s(e, rng.standard_normal((V, 24)).astype(np.float32))
        lib.bnd_s2zero.argtypes = [C.c_int, P]
        lib.bnd_s2zero(0, e)
        eta, zero = lat.get_s(e), np.zeros((V, 24), np.float32)
        out = []
        for prec in (2, 0):
            lib.oqh_set_sap_prec(prec)
            lat.put_s(p, zero)
            lat.put_s(r, eta)
            for _ in range(2):
                lib.sap(0.05, isolv, 4, p, r)
            out.append((lat.get_s(p).astype(np.float64), lat.get_s(r).astype(np.float64)))
        for name, a, b, tol in (("solution", out[1][0], out[0][0], 2e-6), ("residual", out[1][1], out[0][1], 1e-5)):
            d = np.linalg.norm(a - b) / np.linalg.norm(b)
            print(name, d)
            assert d < tol
    finally:
        lat.lib.oqh_set_sap_prec(0)
        lat.close()
