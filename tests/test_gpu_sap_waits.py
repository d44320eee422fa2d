"""Waits between the work-groups that share a Schwarz block (sap.hip
k_sap_cluster) when they are given up.  The bound on the polls is set so low
that the first wait fails (every kernel then ends normally, with incomplete
sums): the call that ran the cycles reports the error, whether the fields lie
on the device or on the host, host arrays stay as they were, and with the
bound restored the next call neither fails nor differs from an undisturbed
one."""
import ctypes as C

import numpy as np
import pytest

import pyoqh
from helpers import make_oracle

P = C.c_void_p
POLLS = 1 << 22


@pytest.fixture
def lat():
    o, eta, _ = make_oracle((16, 16, 16, 16), (8, 8, 8, 8), bc=3, m0=-0.1, csw=1.77, seed=6)
    lat = pyoqh.Lattice((16, 16, 16, 16), (8, 8, 8, 8), bc=3, m0=-0.1, csw=1.77)
    lat.import_ud(o.ud())
    lat.lib.sap.argtypes = [C.c_float, C.c_int, C.c_int, P, P]
    lat.lib.oqh_set_sap_parms((C.c_int * 4)(8, 8, 8, 8), 1, 4, 2)
    lat.lib.oqh_set_error_mode(0)
    lat.eta = eta
    yield lat
    lat.lib.oqh_set_error_mode(1)
    lat.close()


@pytest.mark.gpu
@pytest.mark.parametrize("host", [False, True])
def test_cycle(lat, host):
    lib, V = lat.lib, lat.V
    eta = lat.eta.astype(np.float32)

    def cycle(polls):
        print("host", host, "polls", polls, flush=True)
        lib.oqh_set_sap_polls(polls)
        psi, rho = np.zeros((V, 24), np.float32), eta.copy()
        if host:
            lib.sap(0.0, 1, 4, psi.ctypes.data_as(P), rho.ctypes.data_as(P))
            return lib.oqh_last_error(None, 0), psi, rho
        p, r = lat.alloc_s(), lat.alloc_s()
        lat.put_s(p, psi)
        lat.put_s(r, rho)
        lib.sap(0.0, 1, 4, p, r)
        err = lib.oqh_last_error(None, 0)
        psi, rho = lat.get_s(p), lat.get_s(r)
        lat.free(p)
        lat.free(r)
        return err, psi, rho

    err, psi, rho = cycle(POLLS)
    assert err == 0 and np.linalg.norm(rho) < np.linalg.norm(eta)
    err, psi1, rho1 = cycle(1)
    assert err == 1
    if host:
        assert not psi1.any() and np.array_equal(rho1, eta)
    err, psi2, rho2 = cycle(POLLS)
    assert err == 0 and np.array_equal(psi2, psi) and np.array_equal(rho2, rho)


@pytest.mark.gpu
def test_solve(lat):
    lib = lat.lib
    e, p = lat.alloc_sd(), lat.alloc_sd()
    lat.put_sd(e, lat.eta)

    def solve(polls):
        print("polls", polls, flush=True)
        lib.oqh_set_sap_polls(polls)
        ifail, status = C.c_int(), C.c_int()
        lib.sap_gcr.restype = C.c_double
        lib.sap_gcr.argtypes = [C.c_int, C.c_int, C.c_int, C.c_double, C.c_double, P, P, P, P]
        lib.sap_gcr(8, 64, 0, 1e-8, 0.0, e, p, C.byref(ifail), C.byref(status))
        return lib.oqh_last_error(None, 0), ifail.value, lat.get_sd(p)

    err, ifail, psi = solve(POLLS)
    assert err == 0 and ifail == 0
    err, ifail, _ = solve(1)
    assert err == 1 and ifail == -1
    err, ifail, psi2 = solve(POLLS)
    assert err == 0 and ifail == 0 and np.array_equal(psi2, psi)


@pytest.mark.gpu
def test_subspace_generation(lat):
    lib = lat.lib
    lib.set_dfl_parms((C.c_int * 4)(4, 4, 4, 4), 4)
    lib.set_dfl_pro_parms(16, 256, 1e-2, 24, 1e-2)
    lib.set_dfl_gen_parms(0.13, 0.0, 4, 4, 2)
    lib.start_ranlux(0, 1234)
    ifail, status = (C.c_int * 2)(), (C.c_int * 4)()
    print("polls 1", flush=True)
    lib.oqh_set_sap_polls(1)
    lib.dfl_modes(ifail, status)
    assert lib.oqh_last_error(None, 0) == 1 and ifail[0] == -1
    print("polls", POLLS, flush=True)
    lib.oqh_set_sap_polls(POLLS)
    lib.dfl_modes(ifail, status)
    assert lib.oqh_last_error(None, 0) == 0 and ifail[0] == 0
    lib.oqh_dfl_release()
