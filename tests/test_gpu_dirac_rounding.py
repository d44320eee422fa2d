"""Rounding error of the FP32 operators on small lattices (dirac.hip k_split)
against the FP64 ones on the same FP32 input.  The bounds are what the tile
kernels of larger lattices leave on these fields: the split over eight
wavefronts must not be less precise.  The numbers are sums over 10^5 components,
so they hardly depend on the fields."""
import numpy as np
import pytest

import pyoqh


@pytest.mark.gpu
@pytest.mark.parametrize("op,pset", [("Dw", 3), ("Dwhat", 2)])
@pytest.mark.parametrize("bc,m0,mu,dw,dwhat", [(3, -0.5, 0.0, 6.710e-8, 7.107e-8), (3, -0.3, 0.05, 6.856e-8, 7.266e-8),
                                               (0, -0.3, 0.05, 6.795e-8, 7.169e-8), (0, 0.1, 0.0, 6.782e-8, 6.830e-8)])
def test_rounding(op, pset, bc, m0, mu, dw, dwhat):
    print(op, "bc", bc, "m0", m0, "mu", mu, flush=True)
    lat = pyoqh.Lattice((8, 8, 8, 8), None, bc=bc, m0=m0, csw=1.0 if m0 == -0.5 else 1.77)
    try:
        lib, V = lat.lib, lat.V
        lib.start_ranlux(0, 6)
        lib.random_ud()
        if bc == 3:
            lib.set_ud_phase()
        assert lat.sw_term(pset) == 0
        lib.assign_ud2u()
        lib.assign_swd2sw()
        s, r, sd, rd = lat.alloc_s(), lat.alloc_s(), lat.alloc_sd(), lat.alloc_sd()
        x = np.random.default_rng(6).standard_normal((V, 24)).astype(np.float32)
        lat.put_s(s, x)
        lat.put_sd(sd, x.astype(np.float64))
        mu = float(np.float32(mu))
        getattr(lib, op)(mu, s, r)
        getattr(lib, op + "_dble")(mu, sd, rd)
        n = V if op == "Dw" else V // 2
        a, b = lat.get_s(r)[:n].astype(np.float64), lat.get_sd(rd)[:n]
        d = np.linalg.norm(a - b) / np.linalg.norm(b)
        print("error", d)
        assert d <= (dw if op == "Dw" else dwhat)
    finally:
        lat.close()


@pytest.mark.gpu
@pytest.mark.parametrize("bc", [3, 0])
def test_tiles_twisted_mass(bc):
    """The tile kernels with a twisted mass: Dw, Dwhat and two fields at once, where
    the order in which the compiler fuses the products with the mass and with the
    diagonal shows; the bounds were measured with the better of the two."""
    print("bc", bc, flush=True)
    lat = pyoqh.Lattice((24, 24, 24, 24), (8, 8, 8, 8), bc=bc, m0=-0.3, csw=1.77)
    try:
        lib, V, mu = lat.lib, lat.V, float(np.float32(0.05))
        lib.start_ranlux(0, 6)
        lib.random_ud()
        if bc == 3:
            lib.set_ud_phase()
        s, r, sd, rd = lat.alloc_s(), lat.alloc_s(), lat.alloc_sd(), lat.alloc_sd()
        s2, r2 = lat.alloc_s(), lat.alloc_s()
        x = np.random.default_rng(6).standard_normal((V, 24)).astype(np.float32)
        for op, pset, bound in (("Dw", 3, 6.83e-8), ("Dwhat", 2, 7.22e-8), ("multi", 3, 7.555e-8)):
            assert lat.sw_term(pset) == 0
            lib.assign_ud2u()
            lib.assign_swd2sw()
            lat.put_s(s, x)
            lat.put_s(s2, x)
            lat.put_sd(sd, x.astype(np.float64))
            if op == "multi":
                lib.oqh_Dw_multi(mu, 2, (pyoqh.P * 2)(s2, s), (pyoqh.P * 2)(r2, r))
            else:
                getattr(lib, op)(mu, s, r)
            (lib.Dwhat_dble if op == "Dwhat" else lib.Dw_dble)(mu, sd, rd)
            n = V // 2 if op == "Dwhat" else V
            a, b = lat.get_s(r)[:n].astype(np.float64), lat.get_sd(rd)[:n]
            d = np.linalg.norm(a - b) / np.linalg.norm(b)
            print(op, "error", d)
            assert d <= bound
    finally:
        lat.close()
