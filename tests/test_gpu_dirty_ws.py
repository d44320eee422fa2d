"""The solvers take their workspaces without clearing them and form the
solution update in one pass (linalg.hip k_gcr_solution).  With workspaces
full of NaN a solve gives bit for bit what it gives with cleared ones, for
each Schwarz precision, block kernel and boundary condition; and a short solve
with more Krylov vectors than one update pass takes (32) agrees with the oracle."""
import ctypes as C

import numpy as np
import pytest

import pyoqh
from helpers import make_oracle


def solve(lat, e, p, nkv, nmx, res):
    ifail, status = C.c_int(), C.c_int()
    rho = lat.lib.sap_gcr(nkv, nmx, 0, res, 0.02, e, p, C.byref(ifail), C.byref(status))
    return rho, ifail.value, status.value


@pytest.mark.gpu
@pytest.mark.parametrize("L,bs,prec", [((8, 8, 8, 8), (4, 4, 4, 4), 0), ((8, 8, 8, 8), (4, 4, 4, 4), 1),
                                       ((8, 8, 8, 8), (4, 4, 4, 4), 2), ((16, 8, 8, 8), (8, 4, 4, 4), 0),
                                       ((12, 8, 8, 8), (6, 4, 4, 4), 0)])
@pytest.mark.parametrize("bc", [0, 3])
def test_dirty_workspaces(L, bs, prec, bc):
    print("L", L, "blocks", bs, "prec", prec, "bc", bc, flush=True)
    o, eta, _ = make_oracle(L, bc=bc, m0=-0.1, csw=1.77, seed=5)
    lat = pyoqh.Lattice(L, bc=bc, m0=-0.1, csw=1.77)
    try:
        lat.import_ud(o.ud())
        assert lat.sw_term(3) == 0
        lat.lib.oqh_set_sap_parms((C.c_int * 4)(*bs), 1, 4, 5)
        lat.lib.oqh_set_sap_prec(prec)
        e = lat.alloc_sd()
        lat.put_sd(e, eta)
        p0, p1 = lat.alloc_sd(), lat.alloc_sd()
        first = solve(lat, e, p0, 8, 64, 1e-10)
        assert first[1] == 0
        nan32 = np.full((lat.V, 24), np.nan, np.float32)
        nan64 = np.full((lat.V, 24), np.nan, np.float64)
        lat.lib.reserve_ws.restype = lat.lib.reserve_wsd.restype = C.POINTER(C.c_void_p)
        ws, wsd = lat.lib.reserve_ws(17), lat.lib.reserve_wsd(2)
        for k in range(17):
            lat.put_s(C.c_void_p(ws[k]), nan32)
        for k in range(2):
            lat.put_sd(C.c_void_p(wsd[k]), nan64)
        assert (lat.lib.release_wsd(), lat.lib.release_ws()) == (2, 17)
        again = solve(lat, e, p1, 8, 64, 1e-10)
        assert again == first
        assert np.array_equal(lat.get_sd(p0), lat.get_sd(p1))
    finally:
        lat.lib.oqh_set_sap_prec(0)
        lat.close()


@pytest.mark.gpu
@pytest.mark.parametrize("k", [1, 31, 32, 33, 40])
def test_solution_passes(k):
    # the residual of the solution found is the one that the solver reports
    print("Krylov vectors", k, flush=True)
    L = (8, 8, 8, 8)
    o, eta, _ = make_oracle(L, bc=3, m0=-3.0, csw=1.0, seed=5)
    lat = pyoqh.Lattice(L, bc=3, m0=-3.0, csw=1.0)
    try:
        lat.import_ud(o.ud())
        assert lat.sw_term(3) == 0
        lat.lib.oqh_set_sap_parms((C.c_int * 4)(4, 4, 4, 4), 0, 1, 1)
        e, p = lat.alloc_sd(), lat.alloc_sd()
        lat.put_sd(e, eta)
        rho, ifail, status = solve(lat, e, p, 48, k, 1e-12)
        o.sw_term(3)
        true = np.linalg.norm(eta - o.Dw_dble(0.02, lat.get_sd(p)))
        print("status", status, "residual", rho, "true", true, "of", np.linalg.norm(eta))
        assert status == k and ifail == -1
        # rho is recomputed from psi in FP64 and rounded to FP32 fields
        assert abs(rho - true) <= 1e-6 * true
        # FGCR minimises over the space: k vectors reduce the residual
        assert rho < 0.9 * np.linalg.norm(eta)
    finally:
        lat.close()
