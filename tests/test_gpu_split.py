"""The split kernel of the operators on small lattices (dirac.hip k_split) at
its edges: V/2 no multiple of 64 (even and odd points in one storage block),
V/2 a multiple of 64, the first lattice that is left to the tiles; both
boundary conditions, twisted mass with and without eoflg, links that are not
SU(3), and the zeroing of input and output on the open boundary.  Dw_dble and
Dwhat_dble within 1e-13 per site of the oracle, Dw and Dwhat within 1e-6."""
import numpy as np
import pytest

import pyoqh
from helpers import make_oracle, site_rel


@pytest.mark.gpu
@pytest.mark.parametrize("L,T,bc", [((6, 6, 6, 6), None, 3), ((6, 10, 6, 6), None, 0), ((8, 8, 8, 8), (4, 4, 8, 8), 0),
                                    ((16, 16, 16, 24), (8, 8, 8, 8), 3), ((20, 18, 18, 18), (10, 6, 6, 6), 0)])
@pytest.mark.parametrize("eoflg", [0, 1])
@pytest.mark.parametrize("scale", [1.0, 1.01])
def test_split(L, T, bc, eoflg, scale):
    print("L", L, "bc", bc, "eoflg", eoflg, "links times", scale, flush=True)
    o, eta, s32 = make_oracle(L, T, bc=bc, m0=-0.3, csw=1.77, seed=2, eoflg=eoflg)
    o.set_ud(scale * o.ud())
    o.assign_ud2u()
    lat = pyoqh.Lattice(L, T, bc=bc, m0=-0.3, csw=1.77, eoflg=eoflg)
    try:
        h = lat.V // 2
        lat.import_ud(o.ud())
        # a source that does not vanish on the boundary: Dw zeroes it there
        eta = eta + 0.1
        s32 = (s32 + 0.1).astype(np.float32)
        s, r, sf, rf = lat.alloc_sd(), lat.alloc_sd(), lat.alloc_s(), lat.alloc_s()
        o.sw_term(3)
        o.assign_swd2sw()
        assert lat.sw_term(3) == 0
        lat.put_sd(s, eta)
        lat.put_s(sf, s32)
        e1, s1 = eta.copy(), s32.copy()
        ref, ref32 = o.Dw_dble(0.02, e1), o.Dw(0.02, s1)
        lat.lib.Dw_dble(0.02, s, r)
        lat.lib.Dw(0.02, sf, rf)
        rel, absz = site_rel(lat.get_sd(r), ref)
        assert rel < 1e-13 and absz == 0.0
        assert np.array_equal(lat.get_sd(s), e1)
        rel, absz = site_rel(lat.get_s(rf), ref32)
        assert rel < 1e-6 and absz == 0.0
        assert np.array_equal(lat.get_s(sf), s1)
        o.sw_term(2)
        o.assign_swd2sw()
        assert lat.sw_term(2) == 0
        ref, ref32 = o.Dwhat_dble(0.02, e1.copy())[:h], o.Dwhat(0.02, s1.copy())[:h]
        lat.lib.Dwhat_dble(0.02, s, r)
        lat.lib.Dwhat(0.02, sf, rf)
        rel, absz = site_rel(lat.get_sd(r)[:h], ref)
        assert rel < 1e-13 and absz == 0.0
        rel, absz = site_rel(lat.get_s(rf)[:h], ref32)
        assert rel < 2e-6 and absz == 0.0  # two passes
    finally:
        lat.close()
