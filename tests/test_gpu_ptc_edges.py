"""Weight gradients of the network (ptc.hip k_ptc_wgrad) for every shape of
its matrix tiles -- one, two and four 16x16 tiles, full and padded -- on a
lattice whose points are no multiple of the 128 of a work-group.

With zero weights a single layer's output gradient is -2 e / |e|^2 without
BF16 rounding, so its weight gradient is an FP32 sum of FP32 products and
must agree with complex128 to 1e-5 (384 products per partial sum, 2^-24 each,
in the worst case 2.3e-5 of the sum of moduli, which is the norm's own size
here).  In deeper networks the operands pass through the BF16 mixing of the
other layers: 5e-2 per layer, as for the configured network."""
import ctypes as C

import numpy as np
import pytest

import ptc
import pyoqh
import pyoracle as po
from helpers import link_field

P = C.c_void_p


def ptrs(fields):
    return (C.c_void_p * len(fields))(*fields)


@pytest.mark.gpu
@pytest.mark.parametrize("widths,n,tol", [([4, 4], 1, 1e-5), ([4, 4], 3, 1e-5), ([4, 8, 8, 4], 2, 5e-2),
                                          ([4, 16, 4], 5, 5e-2), ([4, 12, 8, 16, 16, 4], 2, 5e-2),
                                          ([4, 12, 12, 4], 17, 5e-2)])
def test_weight_gradient(widths, n, tol):
    print("widths", widths, "pairs", n, flush=True)
    L = (6, 6, 6, 6)
    o = po.Oracle(L, None, bc=3, m0=-0.35, csw=1.77)
    o.start_ranlux(0, 4)
    o.random_ud()
    iup, idn = o.iupdn()
    U = link_field(o.ud(), iup)
    rng = np.random.default_rng(5)
    Ws = ptc.init_weights(widths, rng)
    if len(widths) == 2:
        Ws = [0 * W for W in Ws]
    lat = pyoqh.Lattice(L, None, bc=3, m0=-0.35, csw=1.77)
    try:
        lat.import_ud(o.ud())
        lib = lat.lib
        w = np.array(widths, np.int32)
        assert lib.oqh_nn_create(len(widths) - 1, w.ctypes.data_as(P)) == 0
        flat = np.ascontiguousarray(np.concatenate([W.ravel() for W in Ws]).view(np.float64))
        lib.oqh_nn_set_weights(flat.ctypes.data_as(P))
        rs = [rng.standard_normal((lat.V, 24)).astype(np.float32) for _ in range(n)]
        es = [(r + rng.standard_normal((lat.V, 24))).astype(np.float32) for r in rs]
        fr, fe = [lat.alloc_s() for _ in range(n)], [lat.alloc_s() for _ in range(n)]
        for k in range(n):
            lat.put_s(fr[k], rs[k])
            lat.put_s(fe[k], es[k])
        if n > 2:
            # a pair without target counts nothing
            es[1] = 0 * es[1]
            lat.put_s(fe[1], es[1])
        dw = np.empty(2 * lib.oqh_nn_nweights())
        loss = lib.oqh_nn_grad(n, ptrs(fr), ptrs(fe), dw.ctypes.data_as(P))
        lo, dref = 0.0, 0.0
        for k in range(n):
            if not es[k].any():
                continue
            acts = ptc.net_fwd(Ws, ptc.spinor_to_field(rs[k]), U, iup, idn)
            l, g = ptc.loss_and_grad(acts[-1], ptc.spinor_to_field(es[k]))
            dW, _ = ptc.net_bwd(Ws, acts, g, U, iup, idn)
            lo += l / n
            dref = dref + np.concatenate([d.ravel() for d in dW]) / n
        got = dw.view(np.complex128)
        assert abs(loss - lo) < min(tol, 2e-2) * lo
        off = 0
        for W in Ws:
            sl = slice(off, off + W.size)
            d = np.linalg.norm(got[sl] - dref[sl]) / np.linalg.norm(dref[sl])
            print("layer", W.shape, "deviation", d)
            assert d < tol
            off += W.size
    finally:
        lat.lib.oqh_nn_free()
        lat.close()


@pytest.mark.gpu
def test_pair_without_target():
    """A pair whose target vanishes counts nothing, whatever its input holds."""
    L, n, widths = (8, 8, 8, 8), 3, np.array([4, 8, 4], np.int32)
    rng = np.random.default_rng(5)
    lat = pyoqh.Lattice(L, None, bc=3)
    try:
        lib = lat.lib
        lib.start_ranlux(0, 4)
        lib.random_ud()
        assert lib.oqh_nn_create(2, widths.ctypes.data_as(P)) == 0
        w = 0.1 * rng.standard_normal(2 * lib.oqh_nn_nweights())
        lib.oqh_nn_set_weights(w.ctypes.data_as(P))
        fr, fe = [lat.alloc_s() for _ in range(n)], [lat.alloc_s() for _ in range(n)]
        for f in fr + fe:
            lat.put_s(f, rng.standard_normal((lat.V, 24)).astype(np.float32))
        lat.put_s(fe[1], np.zeros((lat.V, 24), np.float32))
        out = []
        for x in (0.5, np.inf, np.nan):
            print("input", x, flush=True)
            lat.put_s(fr[1], np.full((lat.V, 24), x, np.float32))
            dw = np.empty_like(w)
            loss = lib.oqh_nn_grad(n, ptrs(fr), ptrs(fe), dw.ctypes.data_as(P))
            out.append((loss, dw))
        for loss, dw in out:
            assert np.isfinite(dw).all() and loss == out[0][0] and np.array_equal(dw, out[0][1])
    finally:
        lat.lib.oqh_nn_free()
        lat.close()
