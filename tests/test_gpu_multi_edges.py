"""Batched operator (dirac.hip k_dw_multi) at the edges of its work split: V/2
no multiple of the 64 pairs of a tile, numbers of fields around the 4 of a
work-group and the 16 of a launch, open and periodic bc, links with and
without a reproducible third row, plain and inverted SW term.  The reference
is the single-field operator on the same state (FP64 1e-14, FP32 1e-6 of the
field's norm: the same terms, rounded in another order)."""
import ctypes as C

import numpy as np
import pytest

import pyoqh

P = C.c_void_p


@pytest.mark.gpu
@pytest.mark.parametrize("L,bc", [((6, 6, 6, 6), 3), ((8, 6, 10, 6), 0)])
@pytest.mark.parametrize("su3", [True, False])
@pytest.mark.parametrize("pset", [3, 2])
@pytest.mark.parametrize("n", [1, 4, 5, 17])
def test_multi_edges(L, bc, su3, pset, n):
    print("L", L, "bc", bc, "su3", su3, "pset", pset, "n", n, flush=True)
    rng = np.random.default_rng(6)
    lat = pyoqh.Lattice(L, None, bc=bc, m0=-0.2, csw=1.77)
    try:
        V = lat.V
        lat.lib.start_ranlux(0, 9)
        lat.lib.random_ud()
        if not su3:
            lat.import_ud(1.01 * lat.export_ud())
        assert lat.sw_term(pset) == 0
        fs = [rng.standard_normal((V, 24)) for _ in range(n)]
        for prec in (64, 32):
            alloc, put, get = ((lat.alloc_sd, lat.put_sd, lat.get_sd) if prec == 64 else
                               (lat.alloc_s, lat.put_s, lat.get_s))
            s, r = [alloc() for _ in range(n)], [alloc() for _ in range(n)]
            one, ref = alloc(), alloc()
            for k in range(n):
                put(s[k], fs[k])
            multi, single = ((lat.lib.oqh_Dw_dble_multi, lat.lib.Dw_dble) if prec == 64 else
                             (lat.lib.oqh_Dw_multi, lat.lib.Dw))
            multi(0.03, n, (P * n)(*s), (P * n)(*r))
            for k in range(n):
                assert np.array_equal(get(s[k]), fs[k].astype(np.float64 if prec == 64 else np.float32))
                put(one, fs[k])
                single(0.03, one, ref)
                a, b = get(r[k]), get(ref)
                assert np.linalg.norm(a - b) <= (1e-14 if prec == 64 else 1e-6) * np.linalg.norm(b)
            for f in s + r + [one, ref]:
                lat.free(f)
    finally:
        lat.close()


@pytest.mark.gpu
@pytest.mark.parametrize("L,prec", [((24, 18, 18, 14), 64), ((26, 22, 22, 22), 32)])
@pytest.mark.parametrize("bc", [3, 0])
@pytest.mark.parametrize("n", [1, 2, 3, 18])
def test_few_fields(L, prec, bc, n):
    """Lattices beyond the split kernel's, where one field takes the tiles of
    the single operator and two take tiles of 128 pairs (V/2 is no multiple of
    them): the inputs stay, also on the boundary points of open bc, where the
    output vanishes."""
    print("L", L, "prec", prec, "bc", bc, "n", n, flush=True)
    rng = np.random.default_rng(8)
    lat = pyoqh.Lattice(L, None, bc=bc, m0=-0.2, csw=1.77)
    try:
        V = lat.V
        lat.lib.start_ranlux(0, 9)
        lat.lib.random_ud()
        assert lat.sw_term(3) == 0
        alloc, put, get = ((lat.alloc_sd, lat.put_sd, lat.get_sd) if prec == 64 else
                           (lat.alloc_s, lat.put_s, lat.get_s))
        fs = rng.standard_normal((V, 24)).astype(np.float64 if prec == 64 else np.float32)
        s, r = [alloc() for _ in range(n)], [alloc() for _ in range(n)]
        one, ref = alloc(), alloc()
        for k in range(n):
            put(s[k], fs * (k + 1))
        put(one, fs)
        multi, single = ((lat.lib.oqh_Dw_dble_multi, lat.lib.Dw_dble) if prec == 64 else
                         (lat.lib.oqh_Dw_multi, lat.lib.Dw))
        multi(0.03, n, (P * n)(*s), (P * n)(*r))
        single(0.03, one, ref)
        b = get(ref)
        for k in range(n):
            assert np.array_equal(get(s[k]), fs * (k + 1))
            a = get(r[k])
            assert not a[(b == 0).all(axis=1)].any()
            assert np.linalg.norm(a - (k + 1) * b) <= (1e-14 if prec == 64 else 1e-6) * np.linalg.norm((k + 1) * b)
    finally:
        lat.close()
