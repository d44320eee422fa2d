"""The little solver at the edges of its work-group counts (dfl.hip: 1024
entries per work-group, sums added by the one that finishes last): one
work-group that is not full, one full one, two, three.  The solution of
ltl_gcr satisfies the little equation formed from the exported blocks of the
operator, to the 1e-10 asked for with a factor 10 for the odd blocks' part."""
import ctypes as C

import numpy as np
import pytest

import pyoqh
from helpers import make_oracle
from test_gpu_dfl import P, _cz, _sig


@pytest.mark.gpu
@pytest.mark.parametrize("L,Ns", [((8, 8, 8, 8), 2), ((8, 8, 8, 16), 40), ((16, 16, 16, 16), 8), ((16, 16, 16, 16), 10),
                                  ((16, 16, 16, 16), 20)])
def test_little_solver(L, Ns):
    print("L", L, "Ns", Ns, flush=True)
    o, eta, _ = make_oracle(L, bc=3, m0=0.1, csw=1.0, seed=3)
    lat = pyoqh.Lattice(L, bc=3, m0=0.1, csw=1.0)
    lib = lat.lib
    _sig(lib)
    try:
        lat.import_ud(o.ud())
        assert lat.sw_term(3) == 0
        bs = np.array((4, 4, 4, 4), np.int32)
        assert lib.set_dfl_parms(bs.ctypes.data_as(P), Ns).Ns == Ns
        lib.set_dfl_pro_parms(6, 64, 1e-10, 8, 1e-2)
        rng = np.random.default_rng(12)
        fm = [lat.alloc_s() for _ in range(Ns)]
        for f in fm:
            lat.put_s(f, rng.standard_normal((lat.V, 24)).astype(np.float32))
        lib.dfl_subspace((P * Ns)(*fm))
        nb = lib.oqh_dfl_blocks(None, None)
        inn, bpts = np.empty((nb, 8), np.int32), np.empty((nb, 256), np.int32)
        lib.oqh_dfl_blocks(inn.ctypes.data_as(P), bpts.ctypes.data_as(P))
        mu = 0.05
        assert lib.set_Awhat(mu) == 0
        e = _cz(rng.standard_normal(nb * Ns) + 1j * rng.standard_normal(nb * Ns))
        x = np.empty(nb * Ns, np.complex128)
        ifail, st = np.zeros(1, np.int32), np.zeros(2, np.int32)
        lib.ltl_gcr(mu, e.ctypes.data_as(P), x.ctypes.data_as(P), ifail.ctypes.data_as(P), st.ctypes.data_as(P))
        lib.set_Aw(mu)
        ablk, ahop = np.empty((nb, Ns, Ns), np.complex128), np.empty((nb, 8, Ns, Ns), np.complex128)
        lib.oqh_dfl_export_Aw(ablk.ctypes.data_as(P), ahop.ctypes.data_as(P))
        xb = x.reshape(nb, Ns)
        y = np.matmul(ablk, xb[:, :, None])[:, :, 0]
        for f in range(8):
            y += np.matmul(ahop[:, f], xb[inn[:, f]][:, :, None])[:, :, 0]
        res = np.linalg.norm(y.reshape(-1) - e) / np.linalg.norm(e)
        print("status", st.tolist(), "residual", res)
        assert ifail[0] == 0 and res < 1e-9
    finally:
        lib.oqh_dfl_release()
        lat.close()
