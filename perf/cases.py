"""Timing cases of the transport engine, through the calls a program makes:
Engine.run_dosxyz (one field), Engine.beamlets_sparse (a dose-influence
matrix), Engine.run_beamlets (batch sums per beamlet) and the serving loop
submit / step / poll.

A case is a dict of plain values:
  call       "field", "dij", "sums" or "serve"
  prec       32 or 64 (the engine's precision)
  phantom    "water", "slab", "patient" or "graded" (a slab phantom with a
             non-uniform grid), n its voxels per axis (patient: across)
  hist       histories per field / beamlet / request; log-uniform up to
             hist_hi where that is given
  batches    statistical batches
  energy     MeV of a monoenergetic source, 0 for the 6 MV spectrum
  charge     -1, 0, 1
  side       field side in cm (field, serve) or of the tiled field (dij, sums)
  bixel      beamlet width in cm; beams gantry angles
  nsplit     photon splitting
  step       True: photons stepped voxel by voxel in the FP32 engine too
             (FP64 always does)
  requests   requests of a serving burst
The seed gives the run's random streams and shifts the field by a few mm.
"""
import ctypes as C
import math

import numpy as np

from ompmc_amd import _native as N, configs as cfg, device as D

DEFAULTS = dict(prec=32, phantom="slab", n=64, hist=100000, hist_hi=0, batches=10, energy=0.0, charge=0, side=10.0,
                bixel=0.5, beams=1, nsplit=1, step=False, requests=1)


def _case(call, **kw):
    return dict(DEFAULTS, call=call, **kw)


def listed():
    return [
        # the smallest call: a check run of a thousand photons in the 40^3
        # water cube; launches and the longest track set its time
        _case("field", name="water_1e3_fp64", prec=64, phantom="water", n=40, hist=1000, energy=2.0, side=5.0),
        # one beamlet request on an idle engine, the unit of interactive
        # planning, in both precisions
        _case("serve", name="beamlet_2e4_fp32", phantom="patient", n=128, hist=20000, bixel=0.5, beams=1),
        _case("serve", name="beamlet_2e4_fp64", prec=64, phantom="patient", n=128, hist=20000, bixel=0.5, beams=1),
        # a clinical electron field: no photon phase, long tracks
        _case("field", name="electrons_2e5_fp32", phantom="water", n=48, hist=200000, energy=6.0, charge=-1),
        # a quick photon field on an odd grid with voxels of unequal size
        # (no delta tracking there)
        _case("field", name="graded_1e6_fp32", phantom="graded", n=61, hist=1000000),
        # photon splitting, the reference's variance reduction
        _case("field", name="split20_1e5_fp32", phantom="water", n=48, hist=100000, energy=6.0, nsplit=20),
        # the FP64 engine on the slab
        _case("field", name="slab_5e6_fp64", prec=64, hist=5000000, batches=50),
        # the headline workload: 1e8 histories on the slab
        _case("field", name="slab_1e8_fp32", hist=100000000, batches=50),
        # a dose-influence matrix of 400 beamlets on the patient phantom
        _case("dij", name="dij_400_fp32", phantom="patient", n=128, hist=10000, hist_hi=1000000),
        # a coarse one in FP64: 25 beamlets of 2 cm
        _case("dij", name="dij_25_fp64", prec=64, phantom="patient", n=95, hist=10000, hist_hi=200000, bixel=2.0),
        # a burst of field requests on three resident phantoms
        _case("serve", name="serve_12_fp32", phantom="mixed", n=0, hist=100000, hist_hi=5000000, requests=12),
        # a plan of five beams on the 256x256x160 phantom
        _case("dij", name="plan_5_beams_fp32", phantom="patient", n=256, hist=4000000, side=8.0, bixel=8.0, beams=5),
    ]


def draw(rng):
    def logint(lo, hi):
        return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    call = rng.choice(["field", "field", "field", "dij", "sums", "serve"])
    prec = rng.choice([32, 32, 64])
    c = dict(prec=prec, batches=rng.choice([2, 5, 10, 20, 50]))
    if call == "field":
        c["phantom"] = rng.choice(["water", "slab", "slab", "patient", "graded"])
        c["n"] = rng.randint(17, 129)
        c["side"] = round(rng.uniform(1.0, 14.0), 2)
        c["energy"] = rng.choice([0.0, round(rng.uniform(1.0, 12.0), 2)])
        c["charge"] = rng.choice([0, 0, 0, -1, 1])
        if c["charge"] and not c["energy"]:
            c["energy"] = 6.0
        c["nsplit"] = rng.choice([1, 1, 1, 5, 20]) if not c["charge"] else 1
        c["step"] = rng.random() < 0.25
        hi = 20000000 if prec == 32 else 5000000
        if c["charge"]:
            hi //= 16
        c["hist"] = logint(1000, hi // (2 * c["nsplit"] if c["nsplit"] > 1 else 1))
    elif call == "serve":
        c["batches"] = 10
        if rng.random() < 0.4:
            c.update(phantom="patient", n=rng.randint(63, 140), hist=logint(3000, 300000),
                     bixel=round(rng.uniform(0.4, 2.0), 2))
        else:
            c.update(phantom="mixed", n=0, hist=30000, hist_hi=logint(100000, 3000000 if prec == 32 else 600000),
                     requests=rng.randint(2, 10))
    else:
        c["batches"] = min(c["batches"], 20)
        c["phantom"] = "patient"
        c["n"] = rng.randint(47, 140)
        c["beams"] = rng.choice([1, 1, 2, 5])
        c["side"] = 8.0
        c["bixel"] = rng.choice([1.0, 1.6, 2.0, 4.0]) if call == "dij" else 8.0
        nb = c["beams"] * round(c["side"] / c["bixel"]) ** 2
        c["hist"] = logint(1000, 20000)
        c["hist_hi"] = int(min(logint(20000, 1000000), (2e7 if prec == 32 else 4e6) / nb * 3)) + c["hist"]
    return _case(call, **c)


# ----------------------------------------------------------------- set-up --
def _graded(n):
    """The slab's layers on a grid whose voxels grow towards the edges and
    with depth."""
    ph = cfg.slab_phantom(n)
    t = np.linspace(-1.0, 1.0, n + 1)
    ph.xb = 8.0 * (0.6 * t + 0.4 * t ** 3)
    ph.yb = ph.xb.copy()
    s = np.linspace(0.0, 1.0, n + 1)
    ph.zb = 16.0 * (0.7 * s + 0.3 * s ** 2)
    zc = 0.5 * (ph.zb[1:] + ph.zb[:-1])
    layer = np.digitize(zc, [3.0, 9.0, 11.0])
    ph.med[:] = np.array([1, 2, 3, 1], np.int32)[layer][:, None, None]
    ph.rho[:] = np.array([1.0, 0.26, 1.85, 1.0])[layer][:, None, None]
    return ph


def _phantoms(c):
    n = c["n"]
    if c["phantom"] == "mixed":
        return cfg.c4_phantoms()
    if c["phantom"] == "water":
        return [cfg.water_cube(n, 0.25 * n if n != 40 else 20.0)]
    if c["phantom"] == "slab":
        return [cfg.slab_phantom(n)]
    if c["phantom"] == "graded":
        return [_graded(n)]
    if n == 256:
        return [cfg.config_phantom("C5")]
    nz = max(12, (3 * n) // 4)
    return [cfg.patient_phantom(n, n, nz, 32.0 / n)]


class _State:
    """Engine with resident tables and phantoms, and the call's arguments."""

    def __init__(self):
        self.eng = None
        self.own = []

    def __del__(self):
        if self.eng is not None:
            self.eng.close()
        for free, obj in self.own:
            free(C.byref(obj))


def prepare(case, seed):
    c = dict(DEFAULTS, **case)
    rng = np.random.default_rng(seed)
    N.ensure_spinms()
    h = N.host()
    st = _State()
    st.case = c
    st.seed = tuple(int(v) for v in rng.integers(1, 2 ** 31, 2))
    shift = rng.uniform(-0.2, 0.2, 2)
    specs = _phantoms(c)
    tab = N.Tables()
    names = ((C.c_char * 64) * N.MXMED)()
    for i, m in enumerate(specs[0].names):
        names[i].value = m.encode()
    paths = N.default_paths()
    N.check(h.omc_tables_build(C.byref(tab), len(specs[0].names), names, C.byref(paths)))
    st.own.append((h.omc_tables_free, tab))
    st.eng = D.Engine(D.FP64 if c["prec"] == 64 else D.FP32, woodcock=-1 if c["step"] else 0)
    st.eng.upload_media(tab)
    nat, st.pid, st.nreg = [], [], []
    for s in specs:
        ph = s.to_native()
        st.own.append((h.omc_phantom_free, ph))
        reg = N.Regions()
        N.check(h.omc_regions_build(C.byref(reg), C.byref(ph), C.byref(tab), 0.7, 0.01))
        st.own.append((h.omc_regions_free, reg))
        st.pid.append(st.eng.upload_phantom(ph, reg))
        st.nreg.append(reg.nreg)
        nat.append(ph)
    spec = N.Spectrum()
    if c["energy"]:
        h.omc_spectrum_mono(C.byref(spec), c["energy"])
    else:
        e, w = cfg.spectrum_6mv()
        P = C.POINTER(C.c_double)
        e, w = np.ascontiguousarray(e), np.ascontiguousarray(w)
        N.check(h.omc_spectrum_from_bins(C.byref(spec), len(e), 0.0, e.ctypes.data_as(P), w.ctypes.data_as(P), 0))

    def field(k, side):
        src = N.SourceDosxyz()
        N.check(h.omc_source_dosxyz_setup(C.byref(src), C.byref(nat[k]), -side / 2 + shift[0], side / 2 + shift[0],
                                          -side / 2 + shift[1], side / 2 + shift[1], 100.0, c["charge"]))
        src.spec = spec
        return src

    def bixels():
        b = cfg.beamlets(gantry_deg=tuple(72.0 * k for k in range(c["beams"])), field=c["side"], bixel=c["bixel"],
                         iso=(float(shift[0]), 0.0, float(shift[1])))
        return N.beamlet_source(spec, b.ibeam, b.src, b.corner, b.side1, b.side2, charge=c["charge"])

    sizes = _sizes(c)
    if c["call"] == "field":
        st.src = field(0, c["side"])
    elif c["call"] in ("dij", "sums"):
        st.src = bixels()
        st.nhist = sizes
        # room for the matrix: a beamlet reaches the voxels of its own width
        # and the scatter around it
        st.cap = int((st.nreg[0] - 1) * len(sizes) * min(0.5, 0.02 * (1.0 + c["bixel"]) ** 2))
    elif c["phantom"] == "mixed":
        pick = np.random.default_rng(4242)          # which phantom and field: the stream's own
        st.reqs = []
        for n in sizes:
            k, side = int(pick.integers(0, 3)), float(pick.uniform(1.0, 15.0))
            src = field(k, side)
            if pick.random() < 0.5:
                h.omc_spectrum_mono(C.byref(src.spec), float(pick.uniform(1.0, 6.0)))
            st.reqs.append((k, src, int(n), 0, 0))
    else:
        src = bixels()
        st.reqs = [(0, src, int(n), 1, int(src.nbeamlets // 2 + k)) for k, n in enumerate(sizes)]
    return st


def _sizes(c):
    """Histories of each beamlet / request (the same for every seed)."""
    if c["call"] == "field":
        n = 1
    elif c["call"] == "serve":
        n = c["requests"]
    else:
        n = c["beams"] * int(round(c["side"] / c["bixel"])) ** 2
    if c["hist_hi"]:
        return cfg.loguniform_histories(n, c["hist"], c["hist_hi"])
    return np.full(n, c["hist"], dtype=np.int64)


# -------------------------------------------------------------------- run --
def run(st):
    c = st.case
    nb = c["batches"]
    if c["call"] == "field":
        s, s2, _, _ = st.eng.run_dosxyz(st.pid[0], st.src, max(1, c["hist"] // nb), nb, seed=st.seed,
                                        nreg=st.nreg[0], nsplit=c["nsplit"])
        return {"sum": s, "sum2": s2}
    if c["call"] == "dij":
        jcs, irs, vals, _ = st.eng.beamlets_sparse(st.pid[0], st.src, st.nhist, nb, 0.01, seed=st.seed, cap=st.cap)
        # the arrays the matrix was written to, whole: their length does not
        # depend on the number of entries (jcs[-1])
        return {"jcs": jcs, "irs": irs.base, "vals": vals.base}
    if c["call"] == "sums":
        s, s2, _ = st.eng.run_beamlets(st.pid[0], st.src, st.nhist, nb, seed=st.seed)
        return {"sum": s, "sum2": s2}
    tickets = [st.eng.submit(st.pid[k], src, n, nbatch=nb, seed=(st.seed[0], st.seed[1] + i), kind=kind, beamlet=b)
               for i, (k, src, n, kind, b) in enumerate(st.reqs)]
    out = [None] * len(tickets)
    while any(o is None for o in out):
        st.eng.step()
        for i, t in enumerate(tickets):
            if out[i] is None:
                res, s, s2 = st.eng.poll(t, st.nreg[st.reqs[i][0]])
                if res.done:
                    out[i] = {"sum": s, "sum2": s2, "histories": res.nhist}
    return out


def exact(case, seed):
    """The results are Monte Carlo sums over random histories: no 64-bit
    closed form exists for them (the expectation differs from any run by the
    statistical error)."""
    return None


def work(case):
    """Algorithmic bytes: 16 per dose deposit (FP64 read and write), medium
    and density per voxel looked up, and the results once.  The counts per
    history are those the engine reports on the 6 MV slab (31 deposits, 78
    voxel crossings or 4 delta-tracking sites); a primary electron makes
    about 4 times the deposits.  Operations: about 450 per charged-particle
    step, 70 steps per photon history."""
    c = dict(DEFAULTS, **case)
    nh = float(_sizes(c).sum())
    per = 9 if c["prec"] == 64 else 5
    voxel_step = c["prec"] == 64 or c["step"] or c["phantom"] == "graded" or c["nsplit"] > 1
    dep = 31.0 * (4 if c["charge"] else 1) * c["nsplit"]
    cross = (78.0 if voxel_step else 4.4) * c["nsplit"]
    if c["phantom"] == "mixed":
        vox = 64 ** 3
    elif c["n"] == 256:
        vox = 256 * 256 * 160
    elif c["phantom"] == "patient":
        vox = c["n"] ** 2 * max(12, (3 * c["n"]) // 4)
    else:
        vox = c["n"] ** 3
    grids = {"field": 1, "sums": c["beams"], "serve": c["requests"], "dij": 1}[c["call"]]
    return {"bytes": nh * (16 * dep + per * cross) + 16.0 * vox * grids,
            "flops": nh * dep / 31.0 * 70 * 450}
