"""The Gram-Schmidt passes of the solver at the edges of their vector groups
(linalg.hip k_mdot_partial: 12 vectors per pass, the Gram entries only in the
passes that ask for them).  After exactly k Krylov vectors the coefficients of
the two-pass form agree with those of the term-by-term form of fgcr.c up to
their FP32 rounding (k 2^-24 each, amplified by the FP32 non-orthogonality of
the vectors, which the Gram correction bounds): the solution within 1e-6
(measured 9e-8), the residual, which is 4e-6 of the source after 26 vectors,
within 1e-3 (measured 2e-5)."""
import ctypes as C

import numpy as np
import pytest

import pyoqh
from helpers import make_oracle


@pytest.mark.gpu
@pytest.mark.parametrize("k", [1, 2, 12, 13, 14, 25, 26])
def test_gram_schmidt_groups(k):
    print("Krylov vectors", k, flush=True)
    L = (8, 8, 8, 8)
    o, eta, _ = make_oracle(L, bc=3, m0=-0.5, csw=1.77, seed=11)
    lat = pyoqh.Lattice(L, bc=3, m0=-0.5, csw=1.77)
    try:
        lat.import_ud(o.ud())
        assert lat.sw_term(3) == 0
        bs = (C.c_int * 4)(4, 4, 4, 4)
        lat.lib.oqh_set_sap_parms(bs, 0, 1, 1)  # a weak preconditioner: many vectors
        e = lat.alloc_sd()
        lat.put_sd(e, eta)
        out = []
        for orth in (0, 1):
            lat.lib.oqh_set_gcr_orth(orth)
            p = lat.alloc_sd()
            ifail, status = C.c_int(), C.c_int()
            rho = lat.lib.sap_gcr(32, k, 0, 1e-12, 0.0, e, p, C.byref(ifail), C.byref(status))
            assert (ifail.value, status.value) == (-1, k)
            out.append((rho, lat.get_sd(p)))
        (r0, p0), (r1, p1) = out
        d = np.linalg.norm(p1 - p0) / np.linalg.norm(p0)
        print("residuals", r0, r1, "solutions differ by", d)
        assert abs(r1 - r0) <= 1e-3 * r0
        assert d <= 1e-6
    finally:
        lat.lib.oqh_set_gcr_orth(1)
        lat.close()
