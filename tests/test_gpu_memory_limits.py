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


@pytest.mark.gpu
@pytest.mark.parametrize("L", [(8, 8, 8, 8), (6, 6, 6, 10)])
def test_training_batch(L):
    """The weight gradient of eight pairs with workspaces for all of them and
    for two only (the sums over the pairs are rounded in another order, in FP32),
    and without the memory for one: then nothing is returned or changed but
    the error count."""
    print("L", L, flush=True)
    widths, n = np.array([4, 16, 12, 4], np.int32), 8
    rng = np.random.default_rng(4)
    lat = pyoqh.Lattice(L, None, bc=3)
    lib = lat.lib
    try:
        lib.start_ranlux(0, 3)
        lib.random_ud()
        fr, fe = [lat.alloc_s() for _ in range(n)], [lat.alloc_s() for _ in range(n)]
        for f in fr + fe:
            lat.put_s(f, rng.standard_normal((lat.V, 24)).astype(np.float32))
        args = (n, (P * n)(*fr), (P * n)(*fe))
        w = rng.standard_normal(2 * 9 * (64 + 192 + 48)) * 0.1
        grads = []
        for limit in (0, 2 * 400 * (lat.V + 63), 300 * lat.V):  # activations: 384 bytes per point and pair
            print("limit", limit, flush=True)
            assert lib.oqh_nn_create(3, widths.ctypes.data_as(P)) == 0
            assert lib.oqh_nn_nweights() * 2 == w.size
            lib.oqh_nn_set_weights(w.ctypes.data_as(P))
            dw = np.full(w.size, 7.0)
            lib.oqh_set_alloc_max(limit)
            lib.oqh_set_error_mode(0)
            loss = [lib.oqh_nn_grad(*args, dw.ctypes.data_as(P)) for _ in range(2)]
            err = lib.oqh_last_error(None, 0)
            w1 = np.empty_like(w)
            if limit == 0 or limit > 400 * lat.V:
                assert err == 0 and loss[0] == loss[1] > 0.0
                grads.append((loss[0], dw))
            else:
                assert err > 0 and loss == [0.0, 0.0] and (dw == 7.0).all()
                assert lib.oqh_nn_train_step(*args, 1e-3) == 0.0
                lib.oqh_nn_get_weights(w1.ctypes.data_as(P))
                assert np.array_equal(w1, w.astype(np.float32))
            lib.oqh_last_error(None, 0)
        (l0, g0), (l1, g1) = grads
        assert abs(l0 - l1) <= 1e-12 * l0
        assert np.linalg.norm(g0 - g1) <= 1e-6 * np.linalg.norm(g0)
    finally:
        lib.oqh_set_error_mode(1)
        lib.oqh_set_alloc_max(0)
        lib.oqh_nn_free()
        lat.close()


@pytest.mark.gpu
def test_solves_together():
    """Several solves without the face fields of several sources (96 bytes per
    point and source): their Schwarz cycles run one after the other, with the
    same arithmetic."""
    n, L, T = 8, (16, 8, 8, 8), (8, 8, 8, 8)
    o, eta, _ = make_oracle(L, T, bc=3, m0=-0.1, csw=1.77, seed=5)
    lat = pyoqh.Lattice(L, T, bc=3, m0=-0.1, csw=1.77)
    try:
        lib, V = lat.lib, lat.V
        lat.import_ud(o.ud())
        assert lat.sw_term(3) == 0
        lib.oqh_set_sap_parms((C.c_int * 4)(4, 4, 4, 4), 1, 4, 5)
        rng = np.random.default_rng(2)
        src, sol = [lat.alloc_sd() for _ in range(n)], [lat.alloc_sd() for _ in range(n)]
        for f in src:
            lat.put_sd(f, rng.standard_normal((V, 24)))
        out = []
        # dirty Krylov vectors: nothing may be taken from them
        lib.reserve_ws.restype = C.POINTER(P)
        lib.alloc_ws(17 * n)
        ws = lib.reserve_ws(17 * n)
        for k in range(17 * n):
            lat.put_s(P(ws[k]), np.full((V, 24), np.nan, np.float32))
        lib.release_ws()
        for limit in (n * 96 * V - 1, 0):
            print("limit", limit, flush=True)
            lib.oqh_set_alloc_max(limit)
            rho, ifail, status = (C.c_double * n)(), (C.c_int * n)(), (C.c_int * n)()
            lib.sap_gcr_multi(n, 8, 128, 0, 1e-10, 0.0, (P * n)(*src), (P * n)(*sol), rho, ifail, status)
            assert not any(ifail)
            out.append((list(status), [lat.get_sd(f) for f in sol]))
        assert out[0][0] == out[1][0]
        for a, b in zip(out[0][1], out[1][1]):
            assert np.array_equal(a, b)
    finally:
        lib.oqh_set_alloc_max(0)
        lat.close()
