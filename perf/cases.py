"""Performance cases of the library: the calls a lattice program makes through
the C ABI (openqcd-2.4.2_amd/pyoqh.py), from the smallest lattice to the
largest, each with its inputs, its necessary work, the accuracy its data types
allow and an independent evaluation in 64 bits with plain torch.

The library holds one lattice, gauge field and parameter set at a time, as a
program does: prepare() opens it for the first state of a case and the further
states of that case share it; another case closes it.  A state's fields are
device fields of the library, shown to torch in place (site-block layout,
[blocks of 64 points, 12, 64, re/im])."""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "openqcd-2.4.2_amd"))
import pyoqh  # noqa: E402

P = C.c_void_p
NO_PTS, ODD_PTS, ALL_PTS = 3, 2, 0


def listed():
    return [
        # the operator on the smallest lattice in use (8^4 periodic, random
        # links, m0=-0.5, csw=1): one call is all latency
        dict(name="dw_dble_8", kind="op", op="Dw_dble", L="8x8x8x8", trd="8x8x8x8", bc=3, m0=-0.5, csw=1.0, links=1,
             flow=0, mu=0.0),
        # the operator-throughput workload: 32^3x64, open bc, flowed links
        dict(name="dw_dble_64x32", kind="op", op="Dw_dble", L="64x32x32x32", trd="8x8x8x8", bc=0, m0=-0.3, csw=1.77,
             links=2, flow=20, mu=0.0),
        # the even-odd operator of a CG or HMC solve on a mid-size lattice
        # whose thread blocks are no multiple of 4 (10x6x6x10) and whose
        # parity has no whole number of 64-point blocks per XCD; twisted mass
        dict(name="dwhat_dble_ragged", kind="op", op="Dwhat_dble", L="20x18x18x30", trd="10x6x6x10", bc=3, m0=-0.3,
             csw=1.77, links=3, flow=20, mu=0.01),
        # the 12 spin-colour columns of a propagator, applied at once
        dict(name="dw_multi_12", kind="multi", n=12, prec=64, L="24x24x24x24", trd="8x8x8x8", bc=3, m0=-0.35, csw=1.77,
             links=3, flow=20, mu=0.0),
        # the FP32 preconditioner at the size of the solver workload: 5
        # Schwarz cycles, 4^4 blocks
        dict(name="sap_48_bs4", kind="sap", prec=0, bs="4x4x4x4", isolv=1, nmr=4, ncy=5, L="48x48x48x48",
             trd="8x8x8x8", bc=3, m0=-0.35, csw=1.77, links=3, flow=20),
        # the same with the 8^4 blocks of the mixed-precision configuration,
        # 32^3x64
        dict(name="sap_64x32_bs8", kind="sap", prec=0, bs="8x8x8x8", isolv=1, nmr=4, ncy=5, L="64x32x32x32",
             trd="8x8x8x8", bc=3, m0=-0.35, csw=1.77, links=3, flow=20),
        # a whole plain solve on the smallest lattice (SAP+GCR, FP32 SAP)
        dict(name="solve_8", kind="solve", prec=0, bs="4x4x4x4", isolv=1, nmr=4, ncy=5, nkv=16, nmx=256, res=1e-10,
             L="8x8x8x8", trd="8x8x8x8", bc=3, m0=-0.5, csw=1.0, links=1, flow=0, vectors=3),
        # a whole solve at 32^3x64 near the critical mass with FP16 storage
        # in the preconditioner
        dict(name="solve_64x32_fp16", kind="solve", prec=1, bs="4x4x4x4", isolv=1, nmr=4, ncy=5, nkv=24, nmx=1024,
             res=1e-10, L="64x32x32x32", trd="8x8x8x8", bc=3, m0=-0.35, csw=1.77, links=5, flow=50, vectors=36),
        # a propagator: 12 sources solved together
        dict(name="solve_multi_12", kind="solves", n=12, prec=0, bs="4x4x4x4", isolv=1, nmr=4, ncy=5, nkv=16, nmx=512,
             res=1e-10, L="24x24x24x24", trd="8x8x8x8", bc=3, m0=-0.25, csw=1.77, links=2, flow=50, vectors=10),
        # a deflated solve; the subspace is made once per gauge field
        dict(name="solve_dfl_24", kind="dfl", prec=0, bs="4x4x4x4", isolv=1, nmr=4, ncy=5, nkv=24, nmx=512, res=1e-10,
             dbs="4x4x4x4", Ns=20, L="24x24x24x24", trd="8x8x8x8", bc=3, m0=-0.35, csw=1.77, links=3, flow=50,
             vectors=11),
        # a program that smooths configurations: links in from host memory,
        # 40 steps of the Wilson flow, links out
        dict(name="flow_24", kind="flow", steps=40, eps=0.01, L="24x24x24x24", trd="8x8x8x8", bc=3, m0=0.0, csw=1.0),
        # forward and backward pass of a training step of the learned
        # preconditioner (four layers, 16^4, a batch of 8 pairs)
        dict(name="nn_grad_16", kind="nn", widths="4-12-16-12-4", n=8, L="16x16x16x16", trd="8x8x8x8", bc=3, m0=-0.35,
             csw=1.77, links=1, flow=50),
    ]


def _pick_lattice(rng, unit, lo, hi, even_units=False):
    """Lattice sizes (multiples of unit[mu]; even multiples on request) with
    a volume between lo and hi, spread over its logarithm."""
    target = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    step = [u * (2 if even_units else 1) for u in unit]
    L = list(step)
    for mu in range(4):
        if L[mu] < 8 and 2 * step[mu] <= 12:
            L[mu] = 2 * step[mu]
    while True:
        grow = [mu for mu in range(4) if np.prod(L) // L[mu] * (L[mu] + step[mu]) <= target and L[mu] < 96]
        if not grow:
            return L
        short = min(L[mu] for mu in grow)
        mu = rng.choice([m for m in grow if L[m] <= 1.6 * short])
        L[mu] += step[mu]


def _txt(v):
    return "x".join(str(int(x)) for x in v)


def _phys(rng, L, trd, m0):
    return dict(L=_txt(L), trd=_txt(trd), bc=rng.choice((0, 3)), m0=m0, csw=rng.choice((1.0, 1.77)),
                links=rng.randrange(1, 50), flow=rng.randrange(10, 40))


def draw(rng):
    kind = rng.choice(("op", "op", "op", "op", "multi", "sap", "sap", "sap", "solve", "solve", "solves", "dfl", "flow",
                       "nn"))
    if kind == "op":
        trd = [rng.choice((4, 6, 8, 8, 10, 12)) for _ in range(4)]
        L = _pick_lattice(rng, trd, 4096, 2.1e6)
        return dict(kind=kind, op=rng.choice(("Dw_dble", "Dw", "Dwhat_dble", "Dwhat")), mu=rng.choice((0.0, 0.01)),
                    **_phys(rng, L, trd, rng.uniform(-0.35, 0.1)))
    if kind == "multi":
        n = rng.randrange(2, 17)
        trd = [rng.choice((4, 6, 8, 8)) for _ in range(4)]
        L = _pick_lattice(rng, trd, 4096, 4e6 / n)
        return dict(kind=kind, n=n, prec=rng.choice((32, 64)), mu=rng.choice((0.0, 0.01)),
                    **_phys(rng, L, trd, rng.uniform(-0.35, 0.1)))
    if kind == "sap":
        bs = rng.choice(((4, 4, 4, 4), (4, 4, 4, 4), (6, 6, 6, 6), (8, 8, 8, 8), (8, 4, 4, 4), (4, 6, 6, 6),
                         (8, 8, 4, 4)))
        L = _pick_lattice(rng, bs, 8192, 2.1e6, True)
        return dict(kind=kind, prec=rng.choice((0, 0, 1)), bs=_txt(bs), isolv=rng.choice((0, 1, 1)),
                    nmr=rng.randrange(3, 6), ncy=rng.randrange(3, 7), **_phys(rng, L, [2 * b if b == 4 else b for b in bs],
                                                                              rng.uniform(-0.3, 0.1)))
    if kind in ("solve", "solves", "dfl"):
        bs = (4, 4, 4, 4)
        if kind == "solve":
            bs = rng.choice((bs, bs, (6, 6, 6, 6), (8, 4, 4, 4)))
        L = _pick_lattice(rng, bs, 4096, {"solve": 8e5, "solves": 1.2e5, "dfl": 2e5}[kind], True)
        c = dict(kind=kind, prec=0 if kind == "solves" else rng.choice((0, 1)), bs=_txt(bs), isolv=1, nmr=4, ncy=5,
                 nkv=rng.choice((16, 24)), nmx=512, res=rng.choice((1e-8, 1e-10)), vectors=8,
                 **_phys(rng, L, [2 * b if b == 4 else b for b in bs], rng.uniform(-0.2, 0.1)))
        if kind == "solves":
            c["n"] = rng.randrange(2, 17)
        if kind == "dfl":
            c.update(dbs="4x4x4x4", Ns=rng.choice((8, 12, 16, 20)), m0=rng.uniform(-0.3, -0.1))
        return c
    if kind == "flow":
        trd = [rng.choice((4, 6, 8, 8)) for _ in range(4)]
        L = _pick_lattice(rng, trd, 4096, 3e5)
        return dict(kind=kind, steps=rng.randrange(5, 50), eps=0.01, L=_txt(L), trd=_txt(trd), bc=rng.choice((0, 3)),
                    m0=0.0, csw=1.0)
    L = _pick_lattice(rng, (4, 4, 4, 4), 4096, 7e4, True)
    w = ["4"] + [rng.choice(("4", "8", "12", "16")) for _ in range(rng.randrange(1, 4))] + ["4"]
    c = dict(kind="nn", widths="-".join(w), n=rng.randrange(2, 9), **_phys(rng, L, (8, 8, 8, 8), rng.uniform(-0.3, 0.0)))
    c["bc"] = 3  # the network knows no boundary rules
    return c


# ---------------------------------------------------------------------------
# the library's state
# ---------------------------------------------------------------------------

_lat = None   # the open lattice
_key = None   # the case it was opened for


def _ints(text):
    return [int(x) for x in text.split("x")]


def _iptr(v):
    a = np.array(v, np.int32)
    return a, a.ctypes.data_as(P)


class _Dev:
    """A device field of the library, shown to torch; freed with the last
    tensor that shows it."""

    def __init__(self, lat, prec):
        self.lat = lat
        self.ptr = lat.alloc_sd() if prec == 64 else lat.alloc_s()
        nblk = (lat.V + 63) // 64
        self.__cuda_array_interface__ = {"shape": (nblk, 12, 64, 2), "typestr": "<f8" if prec == 64 else "<f4",
                                         "data": (self.ptr, False), "version": 3}

    def __del__(self):
        if _lat is self.lat:
            self.lat.free(self.ptr)


class _State:
    def __init__(self, lat, case):
        self.lat, self.lib, self.case = lat, lat.lib, case
        self.ptr, self.t = [], []

    def field(self, prec):
        d = _Dev(self.lat, prec)
        self.lat.sync()  # the library clears it on a stream of its own
        self.t.append(torch.as_tensor(d, device="cuda"))
        self.ptr.append(d.ptr)
        return len(self.ptr) - 1

    def gaussian(self, prec, gen):
        """A Gaussian spinor field, zero on the open boundary."""
        k = self.field(prec)
        t = self.t[k]
        t.normal_(0.0, math.sqrt(0.5), generator=gen)
        if self.lat.V % 64:
            t[-1, :, self.lat.V % 64:, :] = 0
        torch.cuda.synchronize()
        (self.lib.bnd_sd2zero if prec == 64 else self.lib.bnd_s2zero)(ALL_PTS, self.ptr[k])
        self.lat.sync()
        return k


_SOLVE_ARGS = [C.c_int, C.c_int, C.c_int, C.c_double, C.c_double, P, P, P, P]
_TYPES = {"bnd_sd2zero": (None, [C.c_int, P]), "bnd_s2zero": (None, [C.c_int, P]),
          "set_s2zero": (None, [C.c_int, C.c_int, P]), "assign_s2s": (None, [C.c_int, C.c_int, P, P]),
          "assign_sd2s": (None, [C.c_int, C.c_int, P, P]), "sap": (None, [C.c_float, C.c_int, C.c_int, P, P]),
          "diff_sd2s": (None, [C.c_int, C.c_int, P, P, P]), "assign_s2sd": (None, [C.c_int, C.c_int, P, P]),
          "sap_gcr": (C.c_double, _SOLVE_ARGS), "dfl_sap_gcr": (C.c_double, _SOLVE_ARGS),
          "set_Awhat": (C.c_int, [C.c_double])}


def _lattice(case):
    """Opens the lattice of a case: geometry, parameters, gauge field, and
    what a program makes once per gauge field (SW term, deflation subspace,
    network)."""
    global _lat, _key
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if _lat is not None and _key == key:
        return _lat
    if _lat is not None:
        old, _lat, _key = _lat, None, None
        if old.lib.oqh_nn_nweights():
            old.lib.oqh_nn_free()
        old.close()
    lat = pyoqh.Lattice(_ints(case["L"]), _ints(case["trd"]), bc=case["bc"], m0=case["m0"], csw=case["csw"])
    lib = lat.lib
    for name, (res, args) in _TYPES.items():
        f = getattr(lib, name)
        f.restype, f.argtypes = res, args
    if "links" in case:
        lib.start_ranlux(0, case["links"])
        lib.random_ud()
        if case["flow"]:
            lib.fwd_euler(case["flow"], 0.01)
        lib.set_ud_phase()
    kind = case["kind"]
    if kind in ("op", "multi"):
        if lib.sw_term(ODD_PTS if case.get("op", "").startswith("Dwhat") else NO_PTS):
            raise RuntimeError("the SW term cannot be inverted")
    if "bs" in case:
        keep, p = _iptr(_ints(case["bs"]))
        lib.oqh_set_sap_parms(p, case["isolv"], case["nmr"], case["ncy"])
        lib.oqh_set_sap_prec(case["prec"])
    if kind == "nn":
        keep, p = _iptr([4, 4, 4, 4])
        lib.oqh_set_sap_parms(p, 1, 4, 5)
        w = [int(x) for x in case["widths"].split("-")]
        keep, p = _iptr(w)
        if lib.oqh_nn_create(len(w) - 1, p):
            raise RuntimeError("oqh_nn_create")
        wt = _weights(case, lib.oqh_nn_nweights())
        lib.oqh_nn_set_weights(wt.ctypes.data_as(P))
    if kind == "dfl":
        keep, p = _iptr(_ints(case["dbs"]))
        lib.set_dfl_parms(p, case["Ns"])
        lib.set_dfl_pro_parms(16, 64, 1e-2, 24, 1e-2)
        lib.set_dfl_gen_parms(1.0 / (2.0 * (4.0 + case["m0"])), 0.0, 6, 4, 4)
        lib.start_ranlux(0, 7)
        ifail, status = np.zeros(2, np.int32), np.zeros(6, np.int32)
        lib.dfl_modes(ifail.ctypes.data_as(P), status.ctypes.data_as(P))
        if ifail[0] or lib.set_Awhat(0.0):
            raise RuntimeError("the deflation subspace cannot be made")
    lat.sync()
    _lat, _key = lat, key
    return lat


def _weights(case, nw):
    return 0.05 * np.random.default_rng(11).standard_normal(2 * nw)


def _haar(V, gen):
    """4V Haar-random SU(3) links in the layout of udfld(), as a host array."""
    dev = gen.device
    z = torch.randn(4 * V, 2, 3, dtype=torch.complex128, device=dev, generator=gen)
    a, b = z[:, 0], z[:, 1]
    a = a / torch.linalg.vector_norm(a, dim=1, keepdim=True)
    b = b - (a.conj() * b).sum(1, keepdim=True) * a
    b = b / torch.linalg.vector_norm(b, dim=1, keepdim=True)
    c = torch.linalg.cross(a, b).conj()
    u = torch.stack((a, b, c), 1).reshape(4 * V, 9)
    return torch.view_as_real(u).reshape(4 * V, 18).cpu().numpy()


def _zero_time_links(case, ipt, ud):
    """Open bc: the time links at x0 = N0-1 vanish (slot 0 of the odd points
    there, slot 1 of the odd points at x0 = 0)."""
    L = _ints(case["L"])
    V = len(ipt)
    x0 = np.empty(V, np.int64)
    x0[ipt] = np.arange(V) // (L[1] * L[2] * L[3])
    v = ud.reshape(V // 2, 8, 18)
    odd = x0[V // 2:]
    v[odd == L[0] - 1, 0] = 0.0
    v[odd == 0, 1] = 0.0


def prepare(case, seed):
    lat = _lattice(case)
    lib, kind = lat.lib, case["kind"]
    gen = torch.Generator("cuda").manual_seed(int(seed))
    s = _State(lat, case)
    if kind == "op":
        prec = 64 if case["op"].endswith("_dble") else 32
        s.gaussian(prec, gen)
        s.field(prec)
        s.call = getattr(lib, case["op"])
    elif kind == "multi":
        n, prec = case["n"], case["prec"]
        for _ in range(n):
            s.gaussian(prec, gen)
        for _ in range(n):
            s.field(prec)
        s.inp, s.out = (P * n)(*s.ptr[:n]), (P * n)(*s.ptr[n:])
        s.call = lib.oqh_Dw_dble_multi if prec == 64 else lib.oqh_Dw_multi
    elif kind == "sap":
        s.gaussian(32, gen)
        s.field(32)
        s.field(32)
    elif kind in ("solve", "dfl"):
        s.gaussian(64, gen)
        s.field(64)
        s.ifail, s.status = np.zeros(2, np.int32), np.zeros(6, np.int32)
    elif kind == "solves":
        n = case["n"]
        for _ in range(n):
            s.gaussian(64, gen)
        for _ in range(n):
            s.field(64)
        s.inp, s.out = (P * n)(*s.ptr[:n]), (P * n)(*s.ptr[n:])
        s.rho, s.ifail, s.status = np.zeros(n), np.zeros(n, np.int32), np.zeros(n, np.int32)
    elif kind == "flow":
        s.ud = _haar(lat.V, gen)
        if case["bc"] == 0:
            _zero_time_links(case, lat.ipt(), s.ud)
        s.res = np.empty_like(s.ud)
    elif kind == "nn":
        _training_pairs(s, gen)
        s.dw = np.zeros(2 * lib.oqh_nn_nweights())
    return s


def _training_pairs(s, gen):
    """The pairs the network is trained on: the residual that five Schwarz
    cycles leave of a Gaussian source, and the error they leave of the
    solution."""
    lat, lib, n = s.lat, s.lib, s.case["n"]
    r, e = [s.field(32) for _ in range(n)], [s.field(32) for _ in range(n)]
    w = _State(lat, s.case)
    psi, phi, phid = w.field(64), w.field(32), w.field(64)
    ifail, status = np.zeros(2, np.int32), np.zeros(6, np.int32)
    for k in range(n):
        eta = w.gaussian(64, gen)
        lib.sap_gcr(24, 512, 0, 1e-8, 0.0, w.ptr[eta], w.ptr[psi], ifail.ctypes.data_as(P), status.ctypes.data_as(P))
        lib.set_s2zero(lat.VT, 2, w.ptr[phi])
        lib.assign_sd2s(lat.VT, 2, w.ptr[eta], s.ptr[r[k]])
        for _ in range(5):
            lib.sap(0.0, 1, 4, w.ptr[phi], s.ptr[r[k]])
        lib.assign_s2sd(lat.VT, 2, w.ptr[phi], w.ptr[phid])
        lib.diff_sd2s(lat.VT, 2, w.ptr[psi], w.ptr[phid], s.ptr[e[k]])
    lat.sync()
    s.inp, s.out = (P * n)(*s.ptr[:n]), (P * n)(*s.ptr[n:])


def run(s):
    c, lib, lat = s.case, s.lib, s.lat
    kind = c["kind"]
    if kind == "op":
        s.call(c["mu"], s.ptr[0], s.ptr[1])
        return s.t[1]
    if kind == "multi":
        s.call(c["mu"], c["n"], s.inp, s.out)
        return s.t[c["n"]:]
    if kind == "sap":
        eta, psi, rho = s.ptr
        lib.set_s2zero(lat.VT, 2, psi)
        lib.assign_s2s(lat.VT, 2, eta, rho)
        for _ in range(c["ncy"]):
            lib.sap(0.0, c["isolv"], c["nmr"], psi, rho)
        return s.t[1:]
    if kind in ("solve", "dfl"):
        call = lib.sap_gcr if kind == "solve" else lib.dfl_sap_gcr
        call(c["nkv"], c["nmx"], 0, c["res"], 0.0, s.ptr[0], s.ptr[1], s.ifail.ctypes.data_as(P),
             s.status.ctypes.data_as(P))
        if s.ifail[0]:
            raise RuntimeError("the solver failed (%d)" % s.ifail[0])
        return s.t[1]
    if kind == "solves":
        lib.sap_gcr_multi(c["n"], c["nkv"], c["nmx"], 0, c["res"], 0.0, s.inp, s.out, s.rho.ctypes.data_as(P),
                          s.ifail.ctypes.data_as(P), s.status.ctypes.data_as(P))
        if s.ifail.any():
            raise RuntimeError("the solver failed")
        return s.t[c["n"]:]
    if kind == "flow":
        lib.oqh_import_ud(s.ud.ctypes.data_as(P))
        lib.fwd_euler(c["steps"], c["eps"])
        lib.oqh_export_ud(s.res.ctypes.data_as(P))
        return s.res
    loss = lib.oqh_nn_grad(c["n"], s.inp, s.out, s.dw.ctypes.data_as(P))
    return [loss, s.dw]


def _cycle(c, V):
    """Bytes and flops of one Schwarz cycle: links, SW matrices, psi and rho
    in and out once, and the faces."""
    bs = _ints(c["bs"])
    size = 0.5 if c["prec"] == 1 and bs == [4, 4, 4, 4] else 1.0
    rbb = 2.0 * sum(1.0 / b for b in bs)
    return V * size * (960 + 288 * rbb), V * ((c["nmr"] + 1) * 2076.0 + 48 if c["isolv"] else c["nmr"] * 2256.0 + 24)


def work(case):
    V = int(np.prod(_ints(case["L"])))
    kind = case["kind"]
    if kind == "op":
        per = {"Dw_dble": 1536, "Dw": 768, "Dwhat_dble": 1344, "Dwhat": 672}[case["op"]]
        return {"bytes": per * V, "flops": (1908 if "hat" in case["op"] else 1920) * V}
    if kind == "multi":
        size = case["prec"] // 32
        return {"bytes": V * size * (576 + 192 * case["n"]), "flops": 1920 * V * case["n"]}
    if kind == "sap":
        b, f = _cycle(case, V)
        return {"bytes": case["ncy"] * b, "flops": case["ncy"] * f}
    if kind in ("solve", "solves", "dfl"):
        # per Krylov vector: the cycles, one FP32 operator, the Gram-Schmidt
        # step against half of the nkv vectors (read twice)
        b, f = _cycle(case, V)
        n = case.get("n", 1) * case["vectors"]
        k = case["nkv"] // 2
        return {"bytes": n * (case["ncy"] * b + V * (768 + 96 * (2 * k + 8))),
                "flops": n * (case["ncy"] * f + V * (1920 + 384 * k))}
    if kind == "flow":
        # the old links read and the new ones written once per step; the
        # force takes 12 products and 6 traces per link
        return {"bytes": 1152 * V * case["steps"], "flops": 4 * V * 12 * 198 * case["steps"]}
    w = [int(x) for x in case["widths"].split("-")]
    b = f = 0.0
    for i, o in zip(w[:-1], w[1:]):
        # forward, input gradient (all but the first layer) and weight
        # gradient: input and output once each, the links once
        b += V * (24.0 * (i + o) + 288) * 3
        f += V * 9 * (3 * 8.0 * i * o * 3 + 66 * 8.0 / 9 * (2 * i + o))
    return {"bytes": case["n"] * b, "flops": case["n"] * f}


def tolerance(case):
    kind = case["kind"]
    if kind in ("op", "multi"):
        # one application differs from 64 bits by 3e-16 (FP64) and 7e-8
        # (FP32); in FP64 the third row of a link may come from the other two
        # (flowed links: 1e-15)
        fp64 = case["prec"] == 64 if kind == "multi" else case["op"].endswith("_dble")
        return {"rel": 4e-15} if fp64 else {"rel": 3e-7}
    if kind == "sap":
        # solution and residual 1.5e-7 and 3.1e-7 in FP32; with FP16 storage,
        # rounded once per cycle, 5e-4 and 1e-3
        return {"rel": 4e-3} if case["prec"] == 1 and case["bs"] == "4x4x4x4" else {"rel": 1.5e-6}
    if kind in ("solve", "solves", "dfl"):
        # two solutions of residual res differ by up to cond(D) res (2e-8 at
        # the lightest mass for 1e-10)
        return {"rel": 1e3 * case["res"]}
    if kind == "flow":
        return {"rel": 1e-14}  # 1e-15 after 40 steps
    return {"rel": 1e-2}  # gradients with BF16 channel mixing: 3e-3


# ---------------------------------------------------------------------------
# the same quantities in 64 bits with torch, from the definitions
# ---------------------------------------------------------------------------

# gamma_mu = [[0, B_mu], [B_mu^+, 0]] in the representation of the library
_B = [[[-1, 0], [0, -1]], [[0, -1j], [-1j, 0]], [[0, -1], [1, 0]], [[-1j, 0], [0, 1j]]]
_MEM = {}


class _Ref:
    """Wilson-Dirac operator of a link field in torch complex128.  Spinors
    are [points, 4, 3] in the library's order (even points first)."""

    def __init__(self, L, ipt, ud, case, dev):
        self.L, self.V, self.h, self.dev, self.case = L, len(ipt), len(ipt) // 2, dev, case
        V, h = self.V, self.h
        lex = np.empty(V, np.int64)
        lex[ipt] = np.arange(V)
        x = np.stack(np.unravel_index(lex, L), 1)
        self.x = x
        up, dn = [], []
        for mu in range(4):
            y = x.copy()
            y[:, mu] = (x[:, mu] + 1) % L[mu]
            up.append(torch.from_numpy(ipt[np.ravel_multi_index(y.T, L)].astype(np.int64)).to(dev))
            y[:, mu] = (x[:, mu] - 1) % L[mu]
            dn.append(torch.from_numpy(ipt[np.ravel_multi_index(y.T, L)].astype(np.int64)).to(dev))
        self.up, self.dn = up, dn
        m = torch.view_as_complex(torch.from_numpy(ud.reshape(h, 8, 9, 2)).to(dev)).reshape(h, 8, 3, 3)
        self.U = []
        for mu in range(4):
            u = torch.empty(V, 3, 3, dtype=torch.complex128, device=dev)
            u[h:] = m[:, 2 * mu]
            u[:h] = m[up[mu][:h] - h, 2 * mu + 1]
            self.U.append(u)
        t = torch.from_numpy(x[:, 0].copy()).to(dev)
        self.t = t
        self.live = torch.ones(V, dtype=torch.bool, device=dev)
        if case["bc"] == 0:
            self.live = (t > 0) & (t < L[0] - 1)
        self.B = torch.tensor(_B, dtype=torch.complex128, device=dev)

    @staticmethod
    def mm(a, b):
        """Products of 3x3 matrices, [n,3,3] each."""
        return (a[:, :, 0, None] * b[:, None, 0, :] + a[:, :, 1, None] * b[:, None, 1, :] +
                a[:, :, 2, None] * b[:, None, 2, :])

    @staticmethod
    def dag(a):
        return a.mH

    @staticmethod
    def mv(u, v):
        """u v on every spin or channel: [n,3,3] and [n,s,3]."""
        ut = u.transpose(1, 2)
        return v[:, :, 0, None] * ut[:, None, 0] + v[:, :, 1, None] * ut[:, None, 1] + v[:, :, 2, None] * ut[:, None, 2]

    def sw(self):
        """The SW term of both Weyl halves, [2, V, 6, 6]."""
        mm, dag, U, up, dn = self.mm, self.dag, self.U, self.up, self.dn
        A = torch.zeros(2, self.V, 2, 3, 2, 3, dtype=torch.complex128, device=self.dev)
        for mu in range(4):
            for nu in range(mu + 1, 4):
                # the four leaves, counter-clockwise from x
                q = mm(mm(U[mu], U[nu][up[mu]]), dag(mm(U[nu], U[mu][up[nu]])))
                xm, xn = dn[mu], dn[nu]
                q += mm(U[nu], mm(dag(U[mu][up[nu][xm]]), mm(dag(U[nu][xm]), U[mu][xm])))
                xmn = xm[xn]
                q += mm(mm(dag(U[mu][xm]), dag(U[nu][xmn])), mm(U[mu][xmn], U[nu][xn]))
                q += mm(mm(dag(U[nu][xn]), U[mu][xn]), mm(U[nu][up[mu][xn]], dag(U[mu])))
                F = (q - dag(q)) * 0.125
                for hf in range(2):
                    g = (self.B[mu] @ self.B[nu].mH) if hf == 0 else (self.B[mu].mH @ self.B[nu])
                    for a in range(2):
                        for b in range(2):
                            if g[a, b] != 0:
                                A[hf, :, a, :, b, :] += -0.5 * self.case["csw"] * g[a, b] * F
        A = A.reshape(2, self.V, 6, 6)
        d = torch.full((self.V,), 4.0 + self.case["m0"], dtype=torch.float64, device=self.dev)
        if self.case["bc"] == 0:
            A[:, ~self.live] = 0.0
            d[~self.live] = 1.0
        idx = torch.arange(6, device=self.dev)
        A[:, :, idx, idx] += d[None, :, None]
        return A

    def make_sw(self, invert_odd):
        self.A = self.sw()
        if invert_odd:
            self.Ainv = torch.empty_like(self.A[:, self.h:])
            for k in range(2):
                for i in range(0, self.h, 1 << 18):
                    self.Ainv[k, i:i + (1 << 18)] = torch.linalg.inv(self.A[k, self.h + i:min(self.V, self.h + i + (1 << 18))])

    def diag(self, A, s, mu=0.0):
        """(A + i mu gamma5) s with the matrices of the points of s."""
        n = len(s)
        o = torch.empty_like(s)
        for hf in range(2):
            v = s[:, 2 * hf:2 * hf + 2].reshape(n, 6)
            w = torch.zeros_like(v)
            for j in range(6):
                w += A[hf, :, :, j] * v[:, j, None]
            o[:, 2 * hf:2 * hf + 2] = (w + (1j * mu if hf == 0 else -1j * mu) * v).reshape(n, 2, 3)
        return o

    def hop(self, s, par, keep=None):
        """The hopping terms into the points of parity par (0 even, 1 odd)
        from the field s of the other parity.  keep(mu, fwd): which of the
        neighbours count."""
        h = self.h
        pts, src = (slice(h, self.V), 0) if par else (slice(0, h), h)
        acc = torch.zeros(h, 4, 3, dtype=torch.complex128, device=self.dev)
        if self.case["bc"] == 0:
            s = s * self.live[src:src + h, None, None]
        for mu in range(4):
            B = self.B[mu]
            for fwd in (True, False):
                y = (self.up if fwd else self.dn)[mu][pts]
                v = s[y - src]
                if keep is not None:
                    v = v * keep(mu, fwd, pts)[:, None, None]
                sg = -1.0 if fwd else 1.0
                u2 = v[:, :2].clone()
                for a in range(2):
                    for b in range(2):
                        if B[a, b] != 0:
                            u2[:, a] += sg * B[a, b] * v[:, 2 + b]
                w = self.mv(self.U[mu][pts], u2) if fwd else self.mv(self.dag(self.U[mu][y]), u2)
                acc[:, :2] += w
                for a in range(2):
                    for b in range(2):
                        if B[b, a] != 0:
                            acc[:, 2 + a] += sg * B[b, a].conj() * w[:, b]
        if self.case["bc"] == 0:
            acc *= self.live[pts][:, None, None]
        return acc

    def Dw(self, s, mu):
        h = self.h
        r = torch.empty_like(s)
        r[:h] = self.diag(self.A[:, :h], s[:h], mu) - 0.5 * self.hop(s[h:], 0)
        r[h:] = self.diag(self.A[:, h:], s[h:], mu) - 0.5 * self.hop(s[:h], 1)
        return r * self.live[:, None, None]

    def hat(self, s, mu):
        """The even-odd operator on the even half s."""
        h = self.h
        t = self.diag(self.Ainv, -0.5 * self.hop(s, 1))
        return (self.diag(self.A[:, :h], s, mu) + 0.5 * self.hop(t, 0)) * self.live[:h, None, None]

    def solve(self, eta, tol):
        """D^-1 eta by BiCGStab on the even-odd form."""
        h = self.h
        eo = self.diag(self.Ainv, eta[h:])
        b = eta[:h] + 0.5 * self.hop(eo, 0)
        x, r = torch.zeros_like(b), b.clone()
        r0, p, v = r.clone(), torch.zeros_like(b), torch.zeros_like(b)
        rho = al = om = torch.ones((), dtype=torch.complex128, device=self.dev)

        def dot(a, c):
            return (a.conj() * c).sum()

        nb = float(dot(b, b).real) ** 0.5
        for it in range(4000):
            rn = dot(r0, r)
            p = r + (rn / rho) * (al / om) * (p - om * v)
            rho = rn
            v = self.hat(p, 0.0)
            al = rho / dot(r0, v)
            r -= al * v
            t = self.hat(r, 0.0)
            om = dot(t, r) / dot(t, t)
            x += al * p + om * r
            r -= om * t
            if it % 4 == 0:
                res = float(dot(r, r).real) ** 0.5
                if res < tol * nb:
                    break
        xo = eo - self.diag(self.Ainv, -0.5 * self.hop(x, 1))
        return torch.cat((x, xo * self.live[h:, None, None]))

    # ---- Schwarz cycles (multiplicative, two colours, block MinRes) ----

    def sap(self, eta, c):
        h, V, L = self.h, self.V, self.L
        bs = _ints(c["bs"])
        b = self.x // np.array(bs)
        nb = [L[m] // bs[m] for m in range(4)]
        blk = torch.from_numpy(np.ravel_multi_index(b.T, nb).astype(np.int64)).to(self.dev)
        col = torch.from_numpy((b.sum(1) & 1).astype(np.int64)).to(self.dev)
        nblk = int(np.prod(nb))
        same = {}
        for mu in range(4):
            same[mu, True] = blk == blk[self.up[mu]]
            same[mu, False] = blk == blk[self.dn[mu]]

        def inside(mu, fwd, pts):
            return same[mu, fwd][pts]

        def outside(mu, fwd, pts):
            return ~same[mu, fwd][pts]

        def bsum(v, pts):
            return torch.zeros(nblk, dtype=v.dtype, device=self.dev).index_add_(0, blk[pts], v)

        E, O = slice(0, h), slice(h, V)
        A, lv = self.A, self.live
        psi, rho = torch.zeros_like(eta), eta.clone()
        for _ in range(c["ncy"]):
            for k in range(2):
                act = (col == k)[:, None, None]
                s1 = rho * act
                if c["isolv"]:
                    s1[O] = self.diag(self.Ainv, s1[O]) * lv[O, None, None]
                    s1[E] = (s1[E] + 0.5 * self.hop(s1[O], 0, inside)) * lv[E, None, None]
                    pts = E
                else:
                    s1 = s1 * lv[:, None, None]
                    pts = slice(0, V)
                s0 = torch.zeros_like(s1)
                for _mr in range(c["nmr"]):
                    if c["isolv"]:
                        t = self.diag(self.Ainv, -0.5 * self.hop(s1[E], 1, inside))
                        s2 = (self.diag(A[:, E], s1[E]) + 0.5 * self.hop(t, 0, inside)) * lv[E, None, None]
                    else:
                        s2 = torch.empty_like(s1)
                        s2[E] = self.diag(A[:, E], s1[E]) - 0.5 * self.hop(s1[O], 0, inside)
                        s2[O] = self.diag(A[:, O], s1[O]) - 0.5 * self.hop(s1[E], 1, inside)
                        s2 *= lv[:, None, None]
                    rr = bsum((s2.real ** 2 + s2.imag ** 2).sum((1, 2)), pts)
                    z = bsum((s2.conj() * s1[pts]).sum((1, 2)), pts) / torch.where(rr > 0, rr, torch.ones_like(rr))
                    z = z[blk[pts]][:, None, None]
                    s0[pts] += z * s1[pts]
                    s1[pts] -= z * s2
                if c["isolv"]:
                    o = self.diag(self.Ainv, -0.5 * self.hop(s0[E], 1, inside)) * lv[O, None, None]
                    s0[O] = (s1[O] - o) * act[O]
                    s1[O] = 0.0
                psi = psi + s0
                rho = torch.where(act, s1, rho)
                rho[E] += 0.5 * self.hop(s0[O], 0, outside)
                rho[O] += 0.5 * self.hop(s0[E], 1, outside)
        return psi, rho

    # ---- Wilson flow: U <- exp(-eps F) U, F the plaquette force ----

    def flow(self, steps, eps):
        mm, dag, up, dn = self.mm, self.dag, self.up, self.dn
        N0, opn = self.L[0], self.case["bc"] == 0
        eye = torch.eye(3, dtype=torch.complex128, device=self.dev)
        edge = (self.t == 0) | (self.t == N0 - 1)
        for _ in range(steps):
            U = self.U
            F = [torch.zeros_like(u) for u in U]
            for mu in range(4):
                for nu in range(4):
                    if nu == mu:
                        continue
                    w = torch.ones(self.V, dtype=torch.float64, device=self.dev)
                    if opn:
                        w = torch.where(self.t == N0 - 1, 0.0 * w, w) if 0 in (mu, nu) else torch.where(edge, 0.5 * w, w)
                    # the two plaquettes of the plane that start with the link
                    a = mm(mm(U[mu], U[nu][up[mu]]), dag(mm(U[nu], U[mu][up[nu]])))
                    xn = dn[nu]
                    b = mm(mm(U[mu], dag(U[nu][up[mu][xn]])), mm(dag(U[mu][xn]), U[nu][xn]))
                    F[mu] += w[:, None, None] * a + w[xn][:, None, None] * b
            for mu in range(4):
                X = 0.5 * (F[mu] - dag(F[mu]))
                X = X - (X[:, 0, 0] + X[:, 1, 1] + X[:, 2, 2])[:, None, None] / 3.0 * eye
                st = torch.full((self.V,), -eps, dtype=torch.float64, device=self.dev)
                if opn:
                    st = torch.where(self.t == N0 - 1, 0.0 * st, st) if mu == 0 else torch.where(edge, 2.0 * st, st)
                X = X * st[:, None, None]
                ex, term = eye + X, X
                for n in range(2, 16):
                    term = mm(term, X) / n
                    ex = ex + term
                F[mu] = mm(ex, U[mu])
            self.U = F

    def export(self):
        h = self.h
        m = torch.empty(h, 8, 9, dtype=torch.complex128, device=self.dev)
        for mu in range(4):
            m[:, 2 * mu] = self.U[mu][h:].reshape(h, 9)
            m[:, 2 * mu + 1] = self.U[mu][self.dn[mu][h:]].reshape(h, 9)
        return torch.view_as_real(m).reshape(4 * self.V, 18).cpu().numpy()

    # ---- the network ----

    def transports(self, v):
        yield v
        for mu in range(4):
            yield self.mv(self.U[mu], v[self.up[mu]])
            y = self.dn[mu]
            yield self.mv(self.dag(self.U[mu][y]), v[y])

    def network(self, widths, W, v):
        for l in range(len(widths) - 1):
            out = None
            for p, tv in enumerate(self.transports(v)):
                z = (W[l][p] @ tv.permute(1, 0, 2).reshape(widths[l], -1)).reshape(widths[l + 1], self.V, 3)
                out = z if out is None else out + z
            v = out.permute(1, 0, 2)
        return v


def _to_points(t, V):
    """[blocks, 12, 64, 2] -> [V, 4, 3] complex128."""
    z = torch.view_as_complex(t.to(torch.float64).contiguous())
    return z.permute(0, 2, 1).reshape(-1, 12)[:V].reshape(V, 4, 3)


def _to_blocks(z, V):
    n = (V + 63) // 64
    o = torch.zeros(n * 64, 12, dtype=torch.complex128, device=z.device)
    o[:V] = z.reshape(V, 12)
    return torch.view_as_real(o.reshape(n, 64, 12).permute(0, 2, 1).contiguous())


def exact(case, seed):
    V = int(np.prod(_ints(case["L"])))
    kind = case["kind"]
    if kind in ("solve", "solves", "dfl") and V * case.get("n", 1) > 4.2e6:
        return None
    if kind in ("solve", "dfl") and V > 6e5:
        return None
    s = prepare(case, seed)
    lat = s.lat
    dev = torch.device("cuda")
    ud = s.ud if kind == "flow" else lat.export_ud()
    ref = _Ref(_ints(case["L"]), lat.ipt(), ud, case, dev)
    h = V // 2
    if kind == "flow":
        ref.flow(case["steps"], case["eps"])
        return ref.export()
    if kind == "nn":
        w = [int(x) for x in case["widths"].split("-")]
        flat = _weights(case, sum(9 * a * b for a, b in zip(w[:-1], w[1:])))
        flat = torch.view_as_complex(torch.from_numpy(flat.reshape(-1, 2)).to(dev))
        W, o = [], 0
        for i, k in zip(w[:-1], w[1:]):
            W.append(flat[o:o + 9 * i * k].reshape(9, k, i).clone().requires_grad_(True))
            o += 9 * i * k
        total = 0.0
        for k in range(case["n"]):
            r, e = (_to_points(s.t[j], V) for j in (k, case["n"] + k))
            d = ref.network(w, W, r) - e
            loss = (d.real ** 2 + d.imag ** 2).sum() / ((e.real ** 2 + e.imag ** 2).sum() * case["n"])
            loss.backward()
            total += float(loss.detach())
        dw = torch.cat([g.grad.reshape(-1) for g in W])
        return [total, torch.view_as_real(dw).reshape(-1).cpu().numpy()]
    if kind in ("op", "multi"):
        hat = case.get("op", "").startswith("Dwhat")
        ref.make_sw(hat)
        out = []
        for t in s.t[:case.get("n", 1)]:
            v = _to_points(t, V)
            if hat:
                r = torch.zeros_like(v)
                r[:h] = ref.hat(v[:h], case["mu"])
            else:
                r = ref.Dw(v, case["mu"])
            out.append(_to_blocks(r, V))
        return out if kind == "multi" else out[0]
    ref.make_sw(True)
    if kind == "sap":
        psi, rho = ref.sap(_to_points(s.t[0], V), case)
        return [_to_blocks(psi, V), _to_blocks(rho, V)]
    out = [_to_blocks(ref.solve(_to_points(t, V), 1e-13), V) for t in s.t[:case.get("n", 1)]]
    return out if kind == "solves" else out[0]
