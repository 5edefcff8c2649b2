"""Performance cases of the emit-and-propagate path.

Each case is one call (or one short chain of calls) of srw_amd.srwlpy as a
user's script makes it, on host arrays as SRW's API has them:

* traj     CalcPartTraj: the electron's trajectory through the undulator;
* field    CalcElecFieldSR: the field of one electron on a mesh, by the manual
           (method 0) or the adaptive (method 1) quadrature, with the
           wavefront radius, centre and moments that the call returns;
* batch    CalcElecFieldSRBatch: many independent requests of uneven meshes;
* multi_e  EmitPropMultiE: partially coherent intensity of a Gaussian beam;
* prop     PropagElecField (drift, lens, aperture, resampling) and
           CalcIntFromElecField;
* fft      UtiFFT.

Sizes are those of srw_amd/workloads.py, the tests and bench.py.
"""
import math
import random
from array import array

import numpy as np
import torch

from srw_amd import srwlpy
from srw_amd import workloads as W
from srw_amd.srwlib import SRWLOptA, SRWLOptC, SRWLOptD, SRWLOptL, SRWLParticle, SRWLPrtTrj, SRWLWfr

HALF = 1e-3      # half width of the observation mesh [m]
PER = 0.02       # undulator period [m]


def _field(name, nx, ny, ne, np_traj=10001, nper=100, K=1.5, harm=1, span=0.0, tilt=0, meth=0, prec=0.01):
    return {"name": name, "kind": "field", "nx": nx, "ny": ny, "ne": ne, "np": np_traj, "nper": nper, "K": K,
            "harm": harm, "span": span, "tilt": tilt, "meth": meth, "prec": prec}


def listed():
    return [
        # an electron's orbit through a 100-period undulator: the smallest call
        {"name": "traj_10001", "kind": "traj", "np": 10001, "nper": 100, "K": 1.5},
        # spectrum on axis over the first harmonic, adaptive method: what most scripts compute first
        _field("spectrum_axis", 1, 1, 501, span=0.3, meth=1),
        # the plain one-energy field of a zero-emittance electron
        _field("field_101", 101, 101, 1),
        # the same by the adaptive method
        _field("field_101_adaptive", 101, 101, 1, meth=1),
        # an off-axis, tilted electron (no mirror symmetry) on a ragged mesh, third harmonic, a few energies
        _field("field_tilted", 150, 93, 5, K=1.9, harm=3, span=0.01, tilt=1),
        # time-dependent / spectral input wavefront: 201 energies over +/-5 %
        _field("field_201_cube", 201, 201, 201, span=0.05),
        # many independent requests of uneven size in one call
        {"name": "batch_uneven", "kind": "batch", "n": 48, "meshes": "64 128 256 512", "np": 10001, "nper": 100},
        # partially coherent sum, small mesh through a lens and an aperture
        {"name": "multi_e_64", "kind": "multi_e", "n": 64, "electrons": 128, "np": 10001, "rqmc": 0, "lens": 1},
        # partially coherent sum at the benchmark's mesh, quasi-Monte Carlo draws, 30 m drift
        {"name": "multi_e_512", "kind": "multi_e", "n": 512, "electrons": 256, "np": 10001, "rqmc": 1, "lens": 0},
        # one drift of a well sampled wavefront
        {"name": "prop_drift_1024", "kind": "prop", "nx": 1024, "ny": 1024, "ne": 1, "mode": 2, "pm": 1.0, "pd": 1.0,
         "lens": 0, "ap": 0, "inten": 0},
        # a short beamline: resampling, lens, aperture, drifts, intensity at the end, several energies
        {"name": "prop_beamline", "kind": "prop", "nx": 200, "ny": 182, "ne": 9, "mode": 1, "pm": 1.5, "pd": 1.5,
         "lens": 1, "ap": 1, "inten": 1},
        # the bare transform at a size that is not a power of two
        {"name": "fft_1050x880", "kind": "fft", "nx": 1050, "ny": 880, "dir": 1},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# even sizes with factors 2, 3, 5, 7, 11, 13 (SRW's own FFT sizes)
def _fft_size(rng, lo, hi):
    while True:
        n = 2 * _logint(rng, lo // 2, hi // 2)
        m = n
        for p in (2, 3, 5, 7, 11, 13):
            while m % p == 0:
                m //= p
        if m == 1:
            return n


def draw(rng):
    kind = rng.choice(["traj", "field", "field", "field", "batch", "multi_e", "prop", "prop", "fft"])
    np_traj = 2 * _logint(rng, 2000, 8000) + 1
    nper = rng.randint(30, 110)
    K = round(rng.uniform(0.5, 2.5), 3)
    if kind == "traj":
        return {"kind": kind, "np": np_traj + rng.randint(0, 1), "nper": nper, "K": K}
    if kind == "field":
        shape = rng.choice(["axis", "line", "mesh", "mesh", "cube"])
        c = _field("", 1, 1, 1, np_traj=np_traj, nper=nper, K=K, harm=rng.randint(1, 5),
                   span=round(rng.uniform(0.005, 0.06), 4), tilt=rng.randint(0, 1))
        del c["name"]
        if shape == "axis":
            c["ne"] = _logint(rng, 20, 1500)
            c["meth"] = rng.randint(0, 1)
        elif shape == "line":
            c["nx" if rng.random() < 0.5 else "ny"] = _logint(rng, 30, 1000)
            c["ne"] = _logint(rng, 1, 60)
        elif shape == "mesh":
            c["nx"], c["ny"], c["ne"] = _logint(rng, 12, 600), _logint(rng, 12, 600), _logint(rng, 1, 6)
            if c["nx"] * c["ny"] < 20000:
                c["meth"] = rng.randint(0, 1)
        else:
            c["nx"], c["ny"], c["ne"] = _logint(rng, 40, 210), _logint(rng, 40, 210), _logint(rng, 7, 150)
        return c
    if kind == "batch":
        sizes = sorted(_logint(rng, 40, 500) for _ in range(rng.randint(2, 4)))
        return {"kind": kind, "n": rng.randint(6, 40), "meshes": " ".join(map(str, sizes)), "np": np_traj, "nper": nper}
    if kind == "multi_e":
        n = rng.choice([64, 128, 256, 512])
        e = 16 * _logint(rng, 2, 16)
        return {"kind": kind, "n": n, "electrons": e, "np": min(np_traj, 10001), "rqmc": rng.randint(0, 1),
                "lens": rng.randint(0, 1)}
    if kind == "prop":
        ne = _logint(rng, 1, 12)
        top = 1100 if ne < 3 else 400
        nx, ny = _fft_size(rng, 90, top), _fft_size(rng, 90, top)
        if rng.random() < 0.4:
            nx = ny = rng.choice([128, 256, 512] + ([1024] if ne < 3 else []))
        resample = rng.randint(0, 1)
        return {"kind": kind, "nx": nx, "ny": ny, "ne": ne, "mode": rng.randint(0, 2),
                "pm": round(rng.uniform(1.1, 1.7), 3) if resample else 1.0,
                "pd": round(rng.uniform(1.0, 1.7), 3) if resample else 1.0,
                "lens": rng.randint(0, 1), "ap": rng.randint(0, 1), "inten": rng.randint(0, 1)}
    nx, ny = _fft_size(rng, 60, 2000), _fft_size(rng, 60, 2000)
    if rng.random() < 0.4:
        nx, ny = 2 ** rng.randint(6, 11), 2 ** rng.randint(6, 11)
    return {"kind": kind, "nx": nx, "ny": ny, "dir": rng.choice([1, -1])}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _source(case, rng, tilt):
    """(beam, undulator): the case's source with a little of it varied."""
    beam = W.electron_beam()
    if tilt:
        p = beam.partStatMom1
        p.x, p.y = rng.uniform(-40e-6, 40e-6), rng.uniform(-15e-6, 15e-6)
        p.xp, p.yp = rng.uniform(-8e-6, 8e-6), rng.uniform(-4e-6, 4e-6)
        p.gamma *= 1. + rng.uniform(-1e-3, 1e-3)
    K = case.get("K", 1.5) * (1. + rng.uniform(-0.02, 0.02))
    return beam, K, W.planar_undulator(K, PER, case["nper"])


def _energies(beam, K, harm, span, rng):
    e1 = harm * W.first_harmonic_eV(beam.partStatMom1.gamma, K, PER) * (1. + rng.uniform(-1e-3, 1e-3))
    return e1 * (1. - span), e1 * (1. + span)


def _precision(case):
    prec = W.traj_prec(case["np"], per=PER, nper=case["nper"])
    if case.get("meth", 0) == 1:
        prec[0], prec[1] = 1, case["prec"]
    return prec


def _wfr(beam, ne, e0, e1, nx, ny):
    w = W.wavefront(beam, ne, e0, e1, nx, ny, HALF, HALF, 20.)
    if nx == 1:
        w.mesh.xStart = w.mesh.xFin = 0.
    if ny == 1:
        w.mesh.yStart = w.mesh.yFin = 0.
    return w


def _gauss_wfr(case, rng, seed):
    """A beam-like field at 20 m from its waist: a Gaussian with curvature and
    a few per cent of smooth ripple, vertical component a tenth of it."""
    nx, ny, ne = case["nx"], case["ny"], case["ne"]
    beam, e1 = W.electron_beam(), 2000. * (1. + rng.uniform(-0.02, 0.02))
    w = SRWLWfr()
    w.mesh.ne, w.mesh.nx, w.mesh.ny, w.mesh.zStart = ne, nx, ny, 20.
    w.mesh.eStart, w.mesh.eFin = (e1, e1) if ne == 1 else (0.99 * e1, 1.01 * e1)
    w.mesh.xStart, w.mesh.xFin, w.mesh.yStart, w.mesh.yFin = -HALF, HALF, -HALF, HALF
    w.partBeam = beam
    w.arMomX, w.arMomY = array('d', [0] * (11 * ne)), array('d', [0] * (11 * ne))
    w.Rx = w.Ry = 20.
    w.dRx = w.dRy = 0.5
    w.xc, w.yc = rng.uniform(-2e-6, 2e-6), rng.uniform(-2e-6, 2e-6)
    w.avgPhotEn = 0.5 * (w.mesh.eStart + w.mesh.eFin)
    g = np.random.default_rng(seed)
    x, y = np.linspace(-HALF, HALF, nx), np.linspace(-HALF, HALF, ny)
    sx, sy = rng.uniform(1.6e-4, 2.4e-4), rng.uniform(1.3e-4, 2e-4)
    X, Y = np.meshgrid(x, y)
    amp = 1e4 * np.exp(-X ** 2 / (4 * sx * sx) - Y ** 2 / (4 * sy * sy))
    for _ in range(4):
        kx, ky, p = g.uniform(-2e4, 2e4), g.uniform(-2e4, 2e4), g.uniform(0, 6.28)
        amp = amp * (1. + 0.03 * np.cos(kx * X + ky * Y + p))
    es = np.linspace(w.mesh.eStart, w.mesh.eFin, ne)
    ex = np.empty((ny, nx, ne), np.complex64)
    for k, e in enumerate(es):
        lam = 1.239842e-06 / e
        ex[:, :, k] = amp * np.exp(1j * np.pi / (20. * lam) * ((X - w.xc) ** 2 + (Y - w.yc) ** 2))
    ey = (0.1 * np.exp(0.7j) * ex * (1. + 0.2 * X[:, :, None] / HALF)).astype(np.complex64)
    return w, ex.reshape(-1).view(np.float32), ey.reshape(-1).view(np.float32)


def prepare(case, seed):
    rng = random.Random(seed)
    kind = case["kind"]
    if kind == "traj":
        beam, K, mag = _source(case, rng, 1)
        t = SRWLPrtTrj()
        t.allocate(case["np"])
        p = beam.partStatMom1
        t.partInitCond = SRWLParticle(p.x, p.y, 0., p.xp, p.yp, p.gamma, 1, -1)
        half = 0.5 * case["nper"] * PER + 4 * PER
        t.ctStart, t.ctEnd = -half, half
        return {"kind": kind, "trj": t, "mag": mag, "K": K}
    if kind == "field":
        beam, K, mag = _source(case, rng, case["tilt"])
        e0, e1 = _energies(beam, K, case["harm"], case["span"] if case["ne"] > 1 else 0., rng)
        return {"kind": kind, "wfr": _wfr(beam, case["ne"], e0, e1, case["nx"], case["ny"]), "mag": mag,
                "prec": _precision(case), "K": K}
    if kind == "batch":
        meshes = [int(s) for s in case["meshes"].split()]
        wfrs, mags, Ks = [], [], []
        sizes = [2 * meshes[i % len(meshes)] ** 2 for i in range(case["n"])]
        # the requests' fields side by side in one array per component
        ex, ey = np.zeros(sum(sizes), np.float32), np.zeros(sum(sizes), np.float32)
        at = 0
        for i in range(case["n"]):
            beam = W.electron_beam()
            K = rng.uniform(0.5, 2.5)
            n = meshes[i % len(meshes)]
            e0, _ = _energies(beam, K, rng.randint(1, 5), 0., rng)
            w = SRWLWfr(_arEx=ex[at:at + sizes[i]], _arEy=ey[at:at + sizes[i]], _eStart=e0, _eFin=e0, _ne=1,
                        _xStart=-HALF, _xFin=HALF, _nx=n, _yStart=-HALF, _yFin=HALF, _ny=n, _zStart=20.,
                        _partBeam=beam)
            at += sizes[i]
            wfrs.append(w)
            mags.append(W.planar_undulator(K, PER, case["nper"]))
            Ks.append(K)
        return {"kind": kind, "wfr": wfrs, "mag": mags, "prec": _precision(case), "K": Ks, "ex": ex, "ey": ey}
    if kind == "multi_e":
        n = case["n"]
        beam = W.beam_for_multi_e()
        e1 = W.first_harmonic_eV(beam.partStatMom1.gamma, 1.5, PER) * (1. + rng.uniform(-1e-3, 1e-3))
        w = W.wavefront(beam, 1, e1, e1, n, n, HALF, HALF, 20.)
        if case["lens"]:
            els = [SRWLOptA('r', 'a', 1.2e-3, 0.9e-3), SRWLOptL(12., 12.), SRWLOptD(10.)]
            half = 1.2e-3
        else:
            els = [SRWLOptD(30.)]
            half = 2.5e-3
        opt = SRWLOptC(els, [[0, 0, 1.0, 2, 0, 1.0, 1.0, 1.0, 1.0]] * len(els))
        st = W.stokes_like(w)
        st.mesh.xStart, st.mesh.xFin, st.mesh.yStart, st.mesh.yFin = -half, half, -half, half
        return {"kind": kind, "wfr": w, "mag": W.planar_undulator(1.5, PER, 100), "opt": opt, "stokes": st,
                "prec": W.traj_prec(case["np"]), "electrons": case["electrons"], "rqmc": case["rqmc"],
                "seed": rng.randrange(1, 1 << 30)}
    if kind == "prop":
        w, ex, ey = _gauss_wfr(case, rng, seed)
        p0 = [0, 0, 1.0, case["mode"], 0, 1.0, 1.0, 1.0, 1.0]
        p1 = [0, 0, 1.0, case["mode"], 0, case["pm"], case["pd"], case["pm"], case["pd"]]
        els, props = [], []
        if case["ap"]:
            els.append(SRWLOptA('r', 'a', 1.1e-3, 0.9e-3, 20e-6, -10e-6))
            props.append(p0)
        if case["lens"]:
            els.append(SRWLOptL(9., 11., 5e-6, 0.))
            props.append(p0)
        els.append(SRWLOptD(5.))
        props.append(p1)
        return {"kind": kind, "wfr": w, "ex": ex, "ey": ey, "opt": SRWLOptC(els, props), "case": case,
                "inten": None, "mesh": [w.mesh.xStart, w.mesh.xFin, w.mesh.yStart, w.mesh.yFin],
                "geom": [w.Rx, w.Ry, w.dRx, w.dRy, w.xc, w.yc]}
    g = torch.Generator().manual_seed(seed)
    data = torch.randn(case["ny"] * case["nx"] * 2, generator=g).numpy()
    mesh = [-HALF, 2 * HALF / case["nx"], case["nx"], -0.9 * HALF, 1.8 * HALF / case["ny"], case["ny"]]
    return {"kind": kind, "data": data, "mesh": mesh, "dir": case["dir"], "work": np.empty_like(data)}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def _f32(a):
    return np.frombuffer(a, np.float32) if isinstance(a, array) else a


def _wfr_outputs(w):
    """Field, radius and centre, moments.  The moments are single-precision
    values that the structure keeps in double arrays."""
    n = 11 * w.mesh.ne
    return [_f32(w.arEx), _f32(w.arEy), np.array([w.Rx, w.Ry, w.dRx, w.dRy, w.xc, w.yc]),
            np.array(w.arMomX[:n], np.float32), np.array(w.arMomY[:n], np.float32)]


def run(state):
    kind = state["kind"]
    if kind == "traj":
        t = state["trj"]
        srwlpy.CalcPartTraj(t, state["mag"], [1])
        return [np.frombuffer(getattr(t, k), np.float64) for k in ("arX", "arXp", "arY", "arYp", "arZ", "arZp")]
    if kind == "field":
        srwlpy.CalcElecFieldSR(state["wfr"], 0, state["mag"], state["prec"])
        return _wfr_outputs(state["wfr"])
    if kind == "batch":
        srwlpy.CalcElecFieldSRBatch(state["wfr"], state["mag"], state["prec"])
        ws = state["wfr"]
        return [state["ex"], state["ey"], np.array([[w.Rx, w.Ry, w.dRx, w.dRy, w.xc, w.yc] for w in ws]),
                np.array([w.arMomX for w in ws], np.float32), np.array([w.arMomY for w in ws], np.float32)]
    if kind == "multi_e":
        info = srwlpy.EmitPropMultiE(state["stokes"], state["wfr"], state["mag"], state["opt"], state["prec"],
                                     state["electrons"], _seed=state["seed"], _rqmc=state["rqmc"])
        return [_f32(state["stokes"].arS), info["electrons"]]
    if kind == "prop":
        # the call works in place: each pass starts from a copy of the wavefront
        w, case = state["wfr"], state["case"]
        w.arEx, w.arEy = state["ex"].copy(), state["ey"].copy()
        w.mesh.nx, w.mesh.ny = case["nx"], case["ny"]
        w.mesh.xStart, w.mesh.xFin, w.mesh.yStart, w.mesh.yFin = state["mesh"]
        w.Rx, w.Ry, w.dRx, w.dRy, w.xc, w.yc = state["geom"]
        w.arMomX, w.arMomY = array('d', [0] * (11 * case["ne"])), array('d', [0] * (11 * case["ne"]))
        srwlpy.PropagElecField(w, state["opt"])
        out = _wfr_outputs(w) + [np.array([w.mesh.xStart, w.mesh.xFin, w.mesh.yStart, w.mesh.yFin])]
        if case["inten"]:
            n = w.mesh.nx * w.mesh.ny
            if state["inten"] is None or len(state["inten"]) != n:
                state["inten"] = array('f', bytes(4 * n))
            srwlpy.CalcIntFromElecField(state["inten"], w, 6, 0, 3, w.mesh.eStart, 0, 0)
            out.append(_f32(state["inten"]))
        return out
    np.copyto(state["work"], state["data"])
    mesh = list(state["mesh"])
    srwlpy.UtiFFT(state["work"], mesh, state["dir"])
    return [state["work"], np.array(mesh, dtype=np.float64)]


# ---------------------------------------------------------------------------
# work of one pass
# ---------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "traj":
        # four field evaluations a step, about 60 operations each
        return {"bytes": 48 * case["np"], "flops": 240 * case["np"]}
    if kind == "field":
        n = case["nx"] * case["ny"] * case["ne"]
        # method 0: two complex multiply-adds per point and integration point;
        # method 1: about 800 integration points a point, 45 operations each
        return {"bytes": 16 * n, "flops": 16 * n * case["np"] if case["meth"] == 0 else 45 * 800 * n}
    if kind == "batch":
        meshes = [int(s) for s in case["meshes"].split()]
        n = sum(meshes[i % len(meshes)] ** 2 for i in range(case["n"]))
        return {"bytes": 16 * n, "flops": 16 * n * case["np"]}
    if kind == "multi_e":
        n = case["n"] * case["n"]
        return {"bytes": 4 * n, "flops": 16 * n * case["electrons"] * case["np"]}
    if kind == "prop":
        n0 = case["nx"] * case["ny"] * case["ne"]
        n1 = n0 * (case["pm"] * case["pd"]) ** 2
        return {"bytes": int(16 * (n0 + n1)), "flops": int(2 * 2 * 5 * n1 * math.log2(case["nx"] * case["ny"]))}
    n = case["nx"] * case["ny"]
    return {"bytes": 16 * n, "flops": int(5 * n * math.log2(n))}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits (numpy and torch only)
# ---------------------------------------------------------------------------

PI_SR = 3.141592653590


def _und_field(K, nper, y, z):
    """Vertical field of the planar undulator (cos-symmetric, with SRW's end
    fields) at height y and longitudinal position z; K may be an array."""
    kw = 6.2831853072 / PER
    half = 0.5 * nper * PER
    edge = half + 0.25 * PER
    bm = K / (93.37290417576577 * PER) * np.cosh(kw * y)
    pi2 = 3.1415926535898 ** 2
    p, c4 = 2. * pi2 / (3. * PER * PER), 4. * pi2 / (9. * PER * PER)
    zt = edge - 0.25 * PER
    sl = -1. if math.cos(kw * -zt) < 0 else 1.
    sr = -1. if math.cos(kw * zt) > 0 else 1.
    left = z < -edge
    za = np.where(left, z + edge, z - edge)
    end = kw * bm * za * (1. - c4 * za * za) * np.exp(-p * za * za) * np.where(left, sl, sr)
    b = np.where(np.abs(z) > edge, end, bm * np.cos(kw * z))
    return np.where(np.abs(z) > half + 4 * PER, 0., b)


def _trajectory(K, nper, init, gamma, ct0, ct1, n):
    """Fourth-order Runge-Kutta from ct = 0 both ways; K, init and gamma hold
    one entry per electron.  Returns (n, 5, electrons)."""
    K, gamma = np.asarray(K, float), np.asarray(gamma, float)
    mult = -1.602176462e-19 / (9.10938188e-31 * 2.99792458e+08 * gamma)
    g2 = 1. / gamma ** 2

    def deriv(f):
        zd = np.sqrt(1. - (g2 + f[1] * f[1] + f[3] * f[3]))
        by = _und_field(K, nper, f[2], f[4])
        return np.array([f[1], -mult * zd * by, f[3], 0. * f[3], zd])

    def step(y, h):
        d1 = deriv(y)
        d2 = deriv(y + 0.5 * h * d1)
        d3 = deriv(y + 0.5 * h * d2)
        d4 = deriv(y + h * d3)
        return y + h / 6. * (d1 + d4 + 2. * (d2 + d3))

    ds = (ct1 - ct0) / (n - 1)
    tol = (ct1 - ct0) * 1e-12
    i0 = int(abs((-ct0 + tol) / ds))
    s0 = ct0 + i0 * ds
    out = np.empty((n, 5, len(gamma)))
    y0 = np.array(init, float)
    if s0 < -tol:
        y0 = step(y0, s0)
    for idx, end in ((range(i0, -1, -1), ct0), (range(i0, n), ct1)):
        steps = len(idx) - 1
        y = y0
        h = (end - s0) / steps if steps else 0.
        for k, i in enumerate(idx):
            out[i] = y
            if k < steps:
                y = step(y, h)
    return out


def _coefs(f, h):
    f0, f1, f2, f3, f4, f5 = f
    d1, d2 = 1. / (60. * h), 1. / (24. * h * h)
    d3, d4, d5 = d2 / h, d2 / h ** 2, d2 / (5. * h ** 3)
    return [f2, (3 * f0 - 30 * f1 - 20 * f2 + 60 * f3 - 15 * f4 + 2 * f5) * d1,
            -(f0 - 16 * f1 + 30 * f2 - 16 * f3 + f4) * d2, -(f0 + f1 - 10 * f2 + 14 * f3 - 7 * f4 + f5) * d3,
            (f0 - 4 * (f1 + f3) + 6 * f2 + f4) * d4, (-f0 + 5 * (f1 - f4) + 10 * (f3 - f2) + f5) * d5]


def _interp(crd, ib, s, s0, h, bmult):
    """Coordinate, angle, integral of the squared angle, field and its slope
    at s from the tabulated plane (fifth-order polynomials)."""
    n = len(crd)
    idx = np.clip(((s - s0) / h).astype(np.int64), 0, n - 2)
    off = np.where(idx < 2, 0, np.where(idx < n - 3, idx - 2, np.where(idx < n - 2, idx - 3, idx - 4)))
    r = s - (s0 + h * (off + 2))
    c = _coefs([crd[off + k] for k in range(6)], h)
    q = _coefs([ib[off + k] for k in range(6)], h)

    def poly(a):
        v = a[-1]
        for t in a[-2::-1]:
            v = v * r + t
        return v

    d1 = [k * c[k] for k in range(1, 6)]
    d2 = [k * d1[k] for k in range(1, 5)]
    d3 = [k * d2[k] for k in range(1, 4)]
    return poly(c), poly(d1), poly(q), bmult * poly(d2), bmult * poly(d3)


def _angle_integral(a, h, s_rel):
    """Cumulative Simpson integral of a^2 (its first interval's left value
    taken as 0, as SRW has it), zero at the point s_rel from the start."""
    n1 = len(a) - 1
    mid = np.empty(n1)
    mid[0] = 0.0625 * (5. * a[0] + 15. * a[1] - 5. * a[2] + a[3])
    mid[1:n1 - 1] = 0.0625 * (-a[0:n1 - 2] + 9. * a[1:n1 - 1] + 9. * a[2:n1] - a[3:n1 + 1])
    mid[n1 - 1] = 0.0625 * (a[n1 - 3] - 5. * a[n1 - 2] + 15. * a[n1 - 1] + 5. * a[n1])
    left = a[:-1] ** 2
    left[0] = 0.
    out = np.concatenate([[0.], np.cumsum(0.333333333333 * 0.5 * h * (left + 4. * mid ** 2 + a[1:] ** 2))])
    v = _interp(out, out, np.array([s_rel]), 0., h, 1.)[0][0]
    return out - v


def _edge_terms(xo, zo, yobs, s, ev, g2, beta, kph, act):
    """Far-field end term of the integral and the derivative of the integrand
    at an integration edge."""
    (X, Btx, IBx, Bz, dBz), (Z, Btz, IBz, Bx, dBx) = ev
    inv = 1. / (yobs - s)
    dx, dz = xo - X, zo - Z
    bx, bz = Btx - dx * inv, Btz - dz * inv
    dph = kph * (g2 + bx * bx + bz * bz)
    ph = kph * (s * g2 + IBx + IBz + (dx * dx + dz * dz) * inv)
    od = 1. / dph
    ax, az = bx * inv, bz * inv
    cx, cz, tk = beta * Bz, -beta * Bx, 2. * kph
    d2 = tk * (bx * (cx + ax) + bz * (cz + az))
    dax, daz = (2. * ax + cx) * inv, (2. * az + cz) * inv
    cdx, cdz = beta * dBz, -beta * dBx
    d3 = tk * ((cx + ax) ** 2 + (cz + az) ** 2 + bx * (inv * (2. * bx * inv + cx) + cdx)
               + bz * (inv * (2. * bz * inv + cz) + cdz))
    e = torch.polar(torch.ones_like(ph), ph)
    t2x = (dax - ax * d2 * od) * od
    t2z = (daz - az * d2 * od) * od
    qq = (d2 * od) ** 2
    t3x = (-inv * (3. * dax + cdx) + (3. * dax * d2 + ax * d3) * od - 3. * ax * qq) * od * od
    t3z = (-inv * (3. * daz + cdz) + (3. * daz * d2 + az * d3) * od - 3. * az * qq) * od * od
    ok3 = ((t3x == 0) & (t2x == 0)) | ((t3x != 0) & (t3x.abs() < 0.7 * t2x.abs()))
    rx = act * 1j * od * torch.complex(torch.where(ok3, ax + t3x, ax), t2x) * e
    rz = act * 1j * od * torch.complex(torch.where(ok3, az + t3z, az), t2z) * e
    return rx, rz, torch.complex(dax, ax * dph) * e, torch.complex(daz, az * dph) * e


def _exact_field(w, nper, traj, prec, gamma):
    """Ex, Ey of one wavefront by the composite quadrature on the tabulated
    trajectory, all in 64 bits.  The phase is a sum of a part of (x, s) and a
    part of (y, s), so each energy is a pair of complex matrix products."""
    m = w.mesh
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    np_t = int(prec[4])
    half = 0.5 * nper * PER + 4 * PER
    s0, h_t = -half, 2. * half / (np_t - 1)
    g2, beta = 1. / gamma ** 2, -1.60217646263E-19 / (gamma * 9.1093818872E-31 * 2.99792458E+08)
    X, Xp, Y, Yp = (np.ascontiguousarray(traj[:, k]) for k in range(4))
    ibx, iby = _angle_integral(Xp, h_t, half), _angle_integral(Yp, h_t, half)
    s_fin = s0 + h_t * (np_t - 1)
    n = ((int((s_fin - s0) / prec[1]) >> 1) << 1) + 1
    h = (s_fin - s0) / (n - 1)
    s = s0 + h * np.arange(n)
    s[-1] = s_fin
    px = _interp(X, ibx, s, s0, h_t, -1. / beta)
    py = _interp(Y, iby, s, s0, h_t, 1. / beta)
    wt = np.where(np.arange(n) % 2 == 1, 16., 14.)
    wt[0] = wt[-1] = 7.
    T = lambda a: torch.as_tensor(a, dtype=torch.float64, device=dev)
    xs = T(np.linspace(m.xStart, m.xFin, m.nx))[:, None]
    ys = T(np.linspace(m.yStart, m.yFin, m.ny))[:, None]
    inv = T(1. / (m.zStart - s))
    dx, dy = xs - T(px[0]), ys - T(py[0])
    tx = T(s * g2 + px[2] + py[2]) + dx * dx * inv
    ty = dy * dy * inv
    ax = T(wt) * (T(px[1]) - dx * inv) * inv
    ay = T(wt) * (T(py[1]) - dy * inv) * inv
    norm = math.sqrt(1. / 137.0360411 * w.partBeam.Iavg * 1e9 / 1.602189246E-19)
    ex = torch.empty((m.ny, m.nx, m.ne), dtype=torch.complex128, device=dev)
    ey = torch.empty_like(ex)
    one = torch.ones((), dtype=torch.float64, device=dev)
    edges = []
    for i in (0, -1):
        edges.append((s[i], [tuple(float(v[i]) for v in px), tuple(float(v[i]) for v in py)]))
    for k, e in enumerate(np.linspace(m.eStart, m.eFin, m.ne)):
        kph = PI_SR * 1e6 * 0.80654658 * e
        act = norm * e * 0.80654658E-03
        fx, fy = torch.polar(one.expand_as(tx), kph * tx), torch.polar(one.expand_as(ty), kph * ty)
        vx = (act * h / 15.) * (fy @ (ax * fx).T.contiguous())
        vy = (act * h / 15.) * ((ay * fy) @ fx.T.contiguous())
        for sign, (se, ev) in zip((-1., 1.), edges):
            rx, rz, ddx, ddz = _edge_terms(xs.T, ys, m.zStart, se, ev, g2, beta, kph, act)
            vx = vx + sign * (rx - act * h * h / 15. * ddx)
            vy = vy + sign * (rz - act * h * h / 15. * ddz)
        ex[:, :, k], ey[:, :, k] = vx, vy
    flat = lambda v: torch.view_as_real(v).reshape(-1).cpu().numpy()
    return flat(ex), flat(ey)


def _exact_fft(case, seed):
    """SRW's centred transform: sum over points of f exp(-/+ 2 pi i q r) dx dy."""
    st = prepare(case, seed)
    x0, dx, nx, y0, dy, ny = st["mesh"]
    f = st["data"].astype(np.float64).view(np.complex128).reshape(ny, nx)
    sgn = 1. if st["dir"] > 0 else -1.
    qx, qy = (np.arange(nx) - nx // 2) / (nx * dx), (np.arange(ny) - ny // 2) / (ny * dy)
    t = np.fft.fft2(f) if sgn > 0 else np.fft.ifft2(f) * (nx * ny)
    t = np.fft.fftshift(t) * dx * dy
    t = t * np.exp(-2j * np.pi * sgn * qx * x0) * np.exp(-2j * np.pi * sgn * qy * y0)[:, None]
    return [t.reshape(-1).view(np.float64), np.array([qx[0], 1. / (nx * dx), nx, qy[0], 1. / (ny * dy), ny])]


def exact(case, seed):
    kind = case["kind"]
    if kind == "fft":
        return _exact_fft(case, seed)
    if kind == "traj":
        st = prepare(case, seed)
        t, p = st["trj"], st["trj"].partInitCond
        gam = p.gamma * 0.51099890221e-03 * 1000. / 0.511003414
        y = _trajectory([st["K"]], case["nper"], [[p.x], [p.xp], [p.y], [p.yp], [0.]], [gam], t.ctStart, t.ctEnd,
                        case["np"])[:, :, 0]
        zp = np.sqrt(1. - (1. / gam ** 2 + y[:, 1] ** 2 + y[:, 3] ** 2))
        return [np.ascontiguousarray(y[:, k]) for k in (0, 1, 2, 3, 4)] + [zp]
    # the adaptive method's result depends on its own stopping rule; the
    # multi-electron draws and the resampling rules are the library's own
    if kind not in ("field", "batch") or case.get("meth", 0) != 0:
        return None
    st = prepare(case, seed)
    ws = st["wfr"] if kind == "batch" else [st["wfr"]]
    Ks = st["K"] if kind == "batch" else [st["K"]]
    ps = [w.partBeam.partStatMom1 for w in ws]
    gam = [p.gamma * 0.51099890221e-03 * 1000. / 0.511003414 for p in ps]
    init = [[getattr(p, k) for p in ps] for k in ("x", "xp", "y", "yp")] + [[0.] * len(ps)]
    half = 0.5 * case["nper"] * PER + 4 * PER
    y = _trajectory(Ks, case["nper"], init, gam, -half, half, case["np"])
    out = [_exact_field(w, case["nper"], y[:, :, j], st["prec"], gam[j]) for j, w in enumerate(ws)]
    return [np.concatenate([o[0] for o in out]), np.concatenate([o[1] for o in out]), None, None, None]
