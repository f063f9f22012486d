"""The work that users of this framework have it do, as measurable cases.

Six kinds of work, each through the entry points a program calls:

field   one simulation in an engine.Context: reset, run to the end, read the
        fields, the slab state and the probe series back.  "none" is a plain
        vacuum grid with CPML ends, "linear" a Lorentz slab, "kerr" a Lorentz
        slab with a Kerr term and per-cell eps_inf and omega0.  "tuned" takes
        the tiling that configs.TILING_CONFIG2 names, as bench.py does;
        otherwise the context keeps its defaults.
pic     the same with an electron beam coupled (Boris push, CIC deposit), the
        particles read back too.
sweep   sweep.Scheduler.run_batch over ragged sweep points (two passes each,
        spectra on the device), as a reflection-against-frequency sweep is
        run; with beams in a share of the points.
nl      Solver_Engine.IntegratorNL1D, the reference's default run (Kerr cubic
        on the slab, TFSF sine source), parameter objects built as
        MasterController.__Main__ builds them.
looped  MasterController.LoopedSim's input frequency sweep (Lorentz slab, two
        passes a point, FP64).
step    one time step of the Lorentz loop through BaseFDTD11's per-step
        functions, the way a program that keeps the reference's own loop
        calls them.
"""
import contextlib
import math
import os
import sys

import numpy as np

sys.path.insert(0, os.path.join(os.getcwd(), "py-fdtd_pic_amd"))

C0 = 299792458.0
DZ = 1.5e-6 / 40            # lambda0 / 40
SC = 0.5
DT = SC * DZ / C0
PML = 32
Z0 = 376.730313668
Q_E, M_E = -1.602176634e-19, 9.1093837139e-31
TWO_PI = 2.0 * math.pi


def listed():
    return [
        # a user's smallest call: a short pulse through a thin Lorentz film
        dict(name="short_f64", path="field", n=1000, steps=400, precision="f64", slab="linear", tiling="default"),
        # the plain single run: 2,000 cells, 10,000 steps, a 400-cell Lorentz slab, FP64 (config 1)
        dict(name="plain_f64", path="field", n=2000, steps=10000, precision="f64", slab="linear", tiling="default"),
        # an odd grid in FP32, the pulse partly through the slab at the end
        dict(name="ragged_f32", path="field", n=25013, steps=24001, precision="f32", slab="linear", tiling="default"),
        # the headline run: 65,536 cells, 50,000 steps, Lorentz + Kerr slab, FP32 (config 2)
        dict(name="kerr_f32", path="field", n=65536, steps=50000, precision="f32", slab="kerr", tiling="tuned"),
        # the same grid in FP64, short enough to be checked step by step
        dict(name="kerr_f64", path="field", n=65536, steps=4000, precision="f64", slab="kerr", tiling="default"),
        # a dense beam: 1e6 electrons over 10,000 cells of a 65,536-cell grid (config 3)
        dict(name="beam_dense_f32", path="pic", n=65536, steps=8000, particles=1000000, precision="f32"),
        # a sparse beam in the precision that is checked against the reference
        dict(name="beam_sparse_f64", path="pic", n=6000, steps=1000, particles=40000, precision="f64"),
        # a batched material and frequency sweep: ragged grids, field only (config 4)
        dict(name="sweep_f32", path="sweep", jobs=48, beams=0, n_lo=1000, n_hi=65536, steps=10000, precision="f32"),
        # sweep points that carry beams of 1e4 to 1e5 particles (config 4)
        dict(name="sweep_beams_f32", path="sweep", jobs=12, beams=12, n_lo=1000, n_hi=65536, steps=2000,
             precision="f32"),
        # the reference's own default run: 11,555 cells, 19,250 steps, Kerr cubic
        dict(name="nl_dropin_f64", path="nl", domain=0.7, lo=7000, hi=8000),
        # the reference's reflection against frequency: 20 points, two passes each
        dict(name="looped_f64", path="looped", domain=0.7, lo=7000, hi=8000, points=20),
        # one step through the per-step functions on a grid at the older module's limit
        dict(name="per_step_f64", path="step", domain=0.3),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["field", "field", "field", "field", "pic", "pic", "sweep", "sweep", "nl", "looped", "step"])
    prec = rng.choice(["f32", "f64"])
    if kind == "field":
        n = _log(rng, 1000, 65536)
        slab = rng.choice(["none", "linear", "kerr", "kerr"])
        # a single-precision run is read before its slab has rung out to rounding noise
        top = 50000 if prec == "f64" else min(50000, n + 2500)
        return dict(path="field", n=n, steps=_log(rng, 400, top), precision=prec, slab=slab,
                    tiling=rng.choice(["default", "default", "tuned"]))
    if kind == "pic":
        n = _log(rng, 2000, 65536)
        particles = _log(rng, 10000, 1000000)
        steps = _log(rng, 500, max(1000, min(8000, 8000000000 // (particles + n))))
        return dict(path="pic", n=n, steps=min(steps, 3 * n // 2), particles=particles, precision=prec)
    if kind == "sweep":
        beams = rng.random() < 0.4
        jobs = rng.randint(3, 12 if beams else 48)
        return dict(path="sweep", jobs=jobs, beams=rng.randint(1, jobs) if beams else 0, n_lo=1000,
                    n_hi=_log(rng, 4000, 65536), steps=_log(rng, 500, 2000) if beams else _log(rng, 2000, 10000),
                    precision=prec)
    if kind == "nl":
        lo = rng.randint(7000, 7900)
        return dict(path="nl", domain=round(rng.uniform(0.4, 0.7), 3), lo=lo, hi=lo + rng.randint(20, 100))
    if kind == "looped":
        lo = rng.randint(6000, 7900)
        return dict(path="looped", domain=round(rng.uniform(0.4, 0.7), 3), lo=lo, hi=lo + 100,
                    points=rng.randint(14, 20))
    return dict(path="step", domain=round(rng.uniform(0.15, 0.7), 3))


# ---- parameters -----------------------------------------------------------
def _field_params(case, seed):
    """Parameter dict of a field or pic case: the pulse's centre frequency and
    the slab's material come from the seed."""
    rng = np.random.default_rng([seed, 1])
    n, steps = case["n"], case["steps"]
    slab = case.get("slab", "linear")
    t0 = min(120e-15, 0.2 * steps * DT)     # a short run has a short pulse
    p = dict(N=n, steps=steps, Sc=SC, dz=DZ, pml_width=PML, pml_order=3, pml_R0=1e-8, slab_start=n // 2,
             slab_stop=n // 2, eps_inf=1.5, d_eps=2.0, omega0=TWO_PI * 150e12, gamma=TWO_PI * 5e12, chi3=0.0,
             ade=True, src_cell=100, src_f0=rng.uniform(150e12, 250e12), src_tau=t0 / 4, src_t0=t0,
             src_amp=rng.uniform(0.5, 2.0), probes=[60, n - PML - 10])
    if slab == "linear":
        start = n // 2 if case["path"] == "field" else min(1000, n // 2)
        p.update(slab_start=start, slab_stop=min(start + 400, n - PML - 40), eps_inf=rng.uniform(1.2, 2.0),
                 d_eps=rng.uniform(1.0, 3.0))
    elif slab == "kerr":
        f, r = 20000 * n // 65536, 40000 * n // 65536
        p.update(slab_start=f, slab_stop=r, eps_inf=rng.uniform(1.0, 3.0, r - f), chi3=1e-19, src_amp=1.8e8,
                 omega0=TWO_PI * 150e12 * (1.0 + rng.uniform(-0.05, 0.05, r - f)))
    # a run too short for the pulse to reach what it is to meet has its source nearer
    meets = 30000 * n // 65536 if case["path"] == "pic" else p["slab_start"]
    if t0 / DT + 2 * (meets - 100) > 0.95 * steps:
        src = max(100, meets - max(50, int(0.5 * (0.97 * steps - t0 / DT))))
        if src < p["slab_start"] - 20 or src > p["slab_stop"] + 50:
            p.update(src_cell=src, probes=[src - 40, n - PML - 10])
    return p


def _beam(case, p, seed):
    """x (cells), u = gamma v / c, weight: electrons drifting at 0.1 c over the
    middle of the grid."""
    rng = np.random.default_rng([seed, 2])
    n, k = case["n"], case["particles"]
    lo, hi = 30000 * n // 65536, 40000 * n // 65536
    x = lo + rng.uniform(0.0, hi - lo, k)
    beta = rng.normal(0.0, 1e-3, (k, 3))
    beta[:, 2] += 0.1
    u = beta / np.sqrt(1.0 - np.sum(beta * beta, axis=1))[:, None]
    return x, u, 1e16 * (hi - lo) * DZ / k


def _sweep_params(case, seed):
    rng = np.random.default_rng([seed, 3])
    out = []
    for i in range(case["jobs"]):
        # grid sizes spread evenly over their logarithm, so every seed's batch is the same work
        n = int(round(math.exp(math.log(case["n_lo"]) + (i + 0.5) / case["jobs"] *
                               (math.log(case["n_hi"]) - math.log(case["n_lo"])))))
        chi3 = float(rng.uniform(0.0, 2e-19))
        src = min(100, n // 10)
        p = dict(N=n, steps=case["steps"], Sc=SC, dz=DZ, pml_width=PML, pml_order=3, pml_R0=1e-8,
                 slab_start=n // 2, slab_stop=n // 2 + n // 5, eps_inf=1.5, d_eps=float(rng.uniform(0.5, 3.0)),
                 omega0=TWO_PI * 150e12, gamma=TWO_PI * 5e12, chi3=chi3, ade=True, src_cell=src,
                 src_f0=float(rng.uniform(100e12, 300e12)), src_tau=8e-15, src_t0=24e-15, src_amp=1.8e8,
                 probes=[max(PML + 4, src - 40), n - PML - 10])
        if i < case["beams"]:
            lo = n // 8 * 5
            p["beam"] = dict(seed=seed * 1003 + i, n=int(round(10000 * 10 ** ((i + 0.5) / case["beams"]))), cell_lo=lo,
                             cell_hi=min(lo + n // 8, n - PML - 20), v_drift=0.1 * C0, v_th=1e-3 * C0, density=1e16)
        out.append(p)
    np.random.default_rng(7).shuffle(out)      # large and small grids arrive mixed
    return out


# ---- prepare and run ------------------------------------------------------
class _Held:
    """A prepared context and its simulation, closed with the state."""

    def __init__(self, ctx, sim, fields):
        self.ctx, self.sim, self.fields = ctx, sim, fields


def prepare(case, seed):
    kind = case["path"]
    if kind in ("field", "pic"):
        from fdtd_pic_amd import configs, engine
        p = _field_params(case, seed)
        slab = p["slab_stop"] > p["slab_start"]
        fields = ("E", "H") + (("D", "P") if slab else ())
        if kind == "field":
            ctx = engine.Context(case["precision"])
            if case["tiling"] == "tuned":
                ctx.set_tiling(*configs.TILING_CONFIG2[case["precision"]])
            return dict(path=kind, held=_Held(ctx, ctx.add(engine.physical_spec(p)), fields))
        x, u, w = _beam(case, p, seed)
        # one cell per lane and one step per launch, as bench.py runs a beam
        ctx = engine.Context(case["precision"], K=1, S=1)
        beam = engine.Beam(x, u, Q_E, M_E, w, DT, DZ)
        return dict(path=kind, held=_Held(ctx, ctx.add(engine.physical_spec(p), beam=beam), fields + ("J",)))
    if kind == "sweep":
        return dict(path=kind, precision=case["precision"], params=_sweep_params(case, seed))
    rng = np.random.default_rng([seed, 4])
    if kind == "nl":
        import Environment_Setup
        setup = Environment_Setup.envSetup(9e9, case["domain"], case["lo"], case["hi"], nonLinMed=True)
        return dict(path=kind, setup=setup, domain=case["domain"], chi3=1e-3 * rng.uniform(0.8, 1.2),
                    alpha3=rng.uniform(0.6, 0.8))
    if kind == "looped":
        return dict(path=kind, case=dict(case), freq=3.0037e9 * (1.0 + 1e-7 * rng.uniform()))
    import Environment_Setup
    import MasterController as MC
    P = MC.Params(*Environment_Setup.envSetup(9e9, case["domain"], 7000, 8000, LorMed=True), False, case["domain"],
                  9e9, 20, LorentzMed=True, SineCont=True, TFSF=True)
    V = MC.Variables(P.Nz, P.timeSteps, P.vidInterval, 3)
    C_P = MC.CPML_Params(P.dz)
    C_V = MC.CPML_Variables(P.Nz, P.timeSteps)
    P.CPMLXp = P.CPMLXm = True
    start = _step_inputs(V, P, C_V, C_P, rng)
    return dict(path=kind, V=V, P=P, C_P=C_P, C_V=C_V, start=start)


def _step_inputs(V, P, C_V, C_P, rng):
    """The coefficients as the integrator builds them, and a field state in mid-run."""
    import BaseFDTD11
    import Solver_Engine as SE
    BaseFDTD11.FieldInit(V, P)
    V.UpHyMat, V.UpExMat = BaseFDTD11.EmptySpaceCalc(V, P)
    BaseFDTD11.CPML_FieldInit(V, P, C_V, C_P)
    SE.boundCondManager(V, P, C_V, C_P)
    n, f, r = P.Nz + 1, P.materialFrontEdge, P.materialRearEdge
    start = {}
    for obj, name, scale in ((V, "Ex", 1.0), (V, "Hy", 1 / Z0), (V, "Dx", P.permit_0), (V, "polarisationCurr", P.permit_0),
                             (V, "tempTempVarPol", P.permit_0), (C_V, "psi_Ex", 1e-2), (C_V, "psi_Hy", 1e-4)):
        a = scale * rng.normal(0.0, 1.0, n)
        if scale == P.permit_0:
            a[:f] = 0.0
            a[r:] = 0.0
        start[name] = a
        setattr(obj, name, a.copy())
    return start


@contextlib.contextmanager
def _quiet():
    """The reference's set-up functions print; a program that sweeps does not show it."""
    with open(os.devnull, "w") as null, contextlib.redirect_stdout(null):
        yield


def run(state):
    kind = state["path"]
    if kind in ("field", "pic"):
        h = state["held"]
        h.sim.reset()
        h.ctx.run_all()
        out = {f: h.sim.read(f) for f in h.fields}
        out["probes"] = h.sim.probes()
        if kind == "pic":
            out["x"], out["u"], out["alive"] = h.sim.particles()
        return out
    if kind == "sweep":
        from fdtd_pic_amd import sweep
        sch = sweep.Scheduler(state["precision"])
        try:
            done = sch.run_batch([sweep.Job(i, p) for i, p in enumerate(state["params"])])
        finally:
            sch.close()
        done = sorted(done, key=lambda j: j.id)
        return dict(X=np.array([j.X for j in done]))
    if kind == "nl":
        return _run_nl(state)
    if kind == "looped":
        return _run_looped(state)
    return _run_step(state)


def _run_nl(state):
    import MasterController as MC
    P = MC.Params(*state["setup"], False, state["domain"], 9e9, 20)
    P.vidInterval = 50
    V = MC.Variables(P.Nz, P.timeSteps, P.vidInterval, 10)
    C_P = MC.CPML_Params(P.dz)
    C_V = MC.CPML_Variables(P.Nz, P.timeSteps)
    P.CPMLXp = P.CPMLXm = P.TFSF = P.SineCont = P.nonLinMed = True
    P.FreeSpace = P.LorentzMed = P.Gaussian = False
    P.Periods = 1000
    V.chi3Stat, V.alpha3 = state["chi3"], state["alpha3"]
    with _quiet():
        V, P, C_V, C_P, _, _ = MC.Controller(V, P, C_V, C_P)
    return dict(Ex=V.Ex, Hy=V.Hy, psi_Ex=C_V.psi_Ex, psi_Hy=C_V.psi_Hy, Dx=V.Dx, Port1=V.Port1, Port2=V.Port2,
                Ex_History=V.Ex_History)


def _run_looped(state):
    import Environment_Setup
    import MasterController as MC
    c = state["case"]
    with _quiet():
        P = MC.Params(*Environment_Setup.envSetup(state["freq"], c["domain"], c["lo"], c["hi"]), False, c["domain"],
                      state["freq"], 20, LorentzMed=True, SineCont=True, TFSF=True)
        V = MC.Variables(P.Nz, P.timeSteps, P.vidInterval, 1)
        out = MC.LoopedSim(None, V, P, MC.CPML_Variables(P.Nz, P.timeSteps), MC.CPML_Params(P.dz), False, c["domain"],
                           c["lo"], c["hi"], loop=True, points=c["points"])
    _, ref, anal, objs = out[6]
    last = objs[-1][0]
    return dict(ref=ref, anal=anal, Ex=[o[0].Ex for o in objs], before=[o[0].x1ColBe for o in objs],
                Ex_History=last.Ex_History)


def _run_step(state):
    import BaseFDTD11 as B
    V, P, C_V, C_P = state["V"], state["P"], state["C_V"], state["C_P"]
    for name, a in state["start"].items():
        np.copyto(getattr(C_V if name.startswith("psi") else V, name), a)
    V.polarisationCurr = B.ADE_PolarisationCurrent_Ex(V, P, C_V, C_P, 0)
    V.Ex = B.ADE_ExUpdate(V, P, C_V, C_P)
    C_V.psi_Ex, V.Ex = B.CPML_Psi_e_Update(V, P, C_V, C_P)
    V.Dx = B.ADE_DxUpdate(V, P, C_V, C_P)
    V.Ex = B.ADE_ExCreate(V, P, C_V, C_P)
    V.Hy = B.ADE_HyUpdate(V, P, C_V, C_P)
    C_V.psi_Hy, V.Hy = B.CPML_Psi_m_Update(V, P, C_V, C_P)
    return dict(Ex=V.Ex, Hy=V.Hy, Dx=V.Dx, P=V.polarisationCurr, psi_Ex=C_V.psi_Ex, psi_Hy=C_V.psi_Hy)


# ---- work -----------------------------------------------------------------
def _cell_flops(n, slab, kerr):
    """Per step: two differences and two multiply-adds a cell; a slab cell
    adds its polarisation, D and E (and the cubic's root)."""
    return 6.0 * n + slab * (10.0 + (20.0 if kerr else 0.0))


def work(case):
    kind = case["path"]
    w = 4 if case.get("precision") == "f32" else 8
    if kind in ("field", "pic"):
        p = _field_params(case, 0)
        n, steps, slab = p["N"], p["steps"], p["slab_stop"] - p["slab_start"]
        values = 2 * n + 6 * slab + steps + 8 * 2 * PML
        flops = steps * _cell_flops(n, slab, p["chi3"] > 0)
        nbytes = w * values + 8 * 2 * steps
        if kind == "pic":
            nbytes += case["particles"] * 2 * (4 * w + 4)
            flops += 70.0 * steps * case["particles"]
        return dict(bytes=nbytes, flops=flops)
    if kind == "sweep":
        nbytes = flops = 0.0
        for p in _sweep_params(case, 0):
            n, t, slab = p["N"], p["steps"], p["slab_stop"] - p["slab_start"]
            k = p["beam"]["n"] if "beam" in p else 0
            nbytes += 2 * w * (2 * t + 16 * PML) + w * 4 * slab + 2 * 2 * 256 * 16 + 2 * 16 * 2 * k
            flops += 2 * t * _cell_flops(n, 0, False) + t * (_cell_flops(0, slab, True)) + 2 * t * 70.0 * k
            flops += 4 * t * 256 * 8.0
        return dict(bytes=nbytes, flops=flops)
    if kind == "nl":
        n, t, f, r = _nl_shape(case)
        return dict(bytes=8.0 * (20 * n + 4 * t + (t // 50) * n), flops=t * (6.0 * n + 80.0 * (r - f)))
    if kind == "looped":
        # about 160 cells a wavelength: two passes a point, 1.8 steps for each of lo
        n, t = int(case["domain"] / 6.0e-4) + 1900, int(1.8 * case["hi"])
        return dict(bytes=8.0 * case["points"] * (2 * 20 * n + 4 * t + (t // 50) * n),
                    flops=case["points"] * t * (12.0 * n + 10.0 * n * 0.6))
    n = int(case["domain"] / 8.4e-5) + 4800
    return dict(bytes=8.0 * 16 * n, flops=30.0 * n)


def _nl_shape(case):
    dz = C0 / 9e9 / 350
    n = int(case["domain"] / dz) + 2 * 2100
    return n, int((case["hi"] - 1) * 2.75), int(0.1 / dz) + 2100, n - 1


# ---- the same numbers in 64 bits, by plain numpy --------------------------
def exact(case, seed):
    kind = case["path"]
    if kind in ("field", "pic"):
        p = _field_params(case, seed)
        cost = case["steps"] * (60e-6 + 1.2e-8 * p["N"] + 1e-7 * (p["chi3"] > 0) * (p["slab_stop"] - p["slab_start"]) +
                                1.6e-7 * case.get("particles", 0))
        return None if cost > 20 else _physical(p, _beam(case, p, seed) if kind == "pic" else None)
    if kind == "step":
        return _exact_step(prepare(case, seed))
    # 24 to 96 passes of thousands of steps, or 19,250 steps of a cubic in
    # every cell of the slab: minutes of numpy
    return None


def _pml(n):
    m = np.arange(n + 1, dtype=np.float64)
    s0 = SC * 4.0 * (-math.log(1e-8)) / (2.0 * PML)
    de, dh = np.zeros(n + 1), np.zeros(n + 1)
    left, right = m < PML, m >= n - PML
    de[left], dh[left] = (PML - m[left]) / PML, (PML - m[left] - 0.5) / PML
    de[right] = (m[right] - (n - PML)) / PML
    dh[right] = np.minimum((m[right] + 0.5 - (n - PML)) / PML, 1.0)
    me, mh = de > 0, dh > 0
    me[0] = me[n] = mh[n] = False
    return np.exp(-s0 * de ** 3), np.exp(-s0 * dh ** 3), np.flatnonzero(me), np.flatnonzero(mh)


def _physical(p, beam):
    """E, H, D, P, probe series (J, particles) of the physical model: leapfrog,
    CPML, Lorentz polarisation, Kerr root by Newton's method."""
    n, steps, f, r = p["N"], p["steps"], p["slab_start"], p["slab_stop"]
    ns = r - f
    cell = lambda v: np.full(ns, float(v)) if np.ndim(v) == 0 else np.asarray(v)  # noqa: E731
    eps, w0, de, g, chi3 = cell(p["eps_inf"]), cell(p["omega0"]), cell(p["d_eps"]), p["gamma"], p["chi3"]
    den = 1.0 / DT ** 2 + g / (2.0 * DT)
    A, B, C = (2.0 / DT ** 2 - w0 ** 2) / den, (g / (2.0 * DT) - 1.0 / DT ** 2) / den, de * w0 ** 2 / den
    bE, bH, ie, ih = _pml(n)
    t = np.arange(steps) * DT - p["src_t0"]
    src = p["src_amp"] * np.exp(-(t / p["src_tau"]) ** 2) * np.sin(TWO_PI * p["src_f0"] * t)
    E, H, psE, psH = np.zeros(n + 1), np.zeros(n + 1), np.zeros(len(ie)), np.zeros(len(ih))
    D, P, Pm = np.zeros(ns), np.zeros(ns), np.zeros(ns)
    probes = np.zeros((2, steps))
    if beam is not None:
        x, u, w = np.array(beam[0]), np.array(beam[1]), beam[2]
        alive, Hprev, J = np.ones(len(x), dtype=bool), np.zeros(n + 1), np.zeros(n + 1)
        a, js = Q_E * DT / (2.0 * M_E * C0), Z0 * Q_E * w * C0
    for k in range(steps):
        if beam is not None:
            J = _push(x, u, alive, E, 0.5 * (Hprev + H), a, js, n)
            Hprev = H.copy()
        if ns:
            P, Pm = A * P + B * Pm + C * E[f:r], P
        dH = H[1:n] - H[:n - 1]
        inc = dH - J[1:n] if beam is not None else dH
        E[1:n] += SC * inc
        psE = bE[ie] * psE + (bE[ie] - 1.0) * dH[ie - 1]
        E[ie] += SC * psE
        E[p["src_cell"]] += src[k]
        if ns:
            D += SC * inc[f - 1:r - 1]
            v = D - P
            e = v / eps
            if chi3:
                for _ in range(3):
                    e -= (chi3 * e ** 3 + eps * e - v) / (3.0 * chi3 * e ** 2 + eps)
            E[f:r] = e
        dE = E[1:] - E[:n]
        H[:n] += SC * dE
        psH = bH[ih] * psH + (bH[ih] - 1.0) * dE[ih]
        H[ih] += SC * psH
        probes[:, k] = E[p["probes"]]
    out = dict(E=E, H=H, probes=probes)
    if ns:
        out.update(D=D, P=P)
    if beam is not None:
        out.update(J=J, x=x, u=u, alive=None)
    return out


def _push(x, u, alive, E, H, a, js, n):
    """Boris push of the live particles in place; the CIC current at the half step."""
    J = np.zeros(n + 1)
    on = np.flatnonzero(alive)
    xs, us = x[on], u[on]
    i = np.floor(xs).astype(np.int64)
    fr = xs - i
    Eg = (1.0 - fr) * E[i] + fr * E[i + 1]
    j = np.floor(xs - 0.5).astype(np.int64)
    fr = xs - 0.5 - j
    Hg = (1.0 - fr) * H[j] + fr * H[j + 1]
    us[:, 0] += a * Eg
    ty = -a * Hg / np.sqrt(1.0 + np.sum(us * us, axis=1))
    sy = 2.0 * ty / (1.0 + ty * ty)
    px, pz = us[:, 0] - us[:, 2] * ty, us[:, 2] + us[:, 0] * ty
    us[:, 0], us[:, 2] = us[:, 0] - pz * sy + a * Eg, us[:, 2] + px * sy
    gam = np.sqrt(1.0 + np.sum(us * us, axis=1))
    half = xs + 0.5 * SC * us[:, 2] / gam
    xs = xs + SC * us[:, 2] / gam
    i = np.floor(half).astype(np.int64)
    q, fr = js * us[:, 0] / gam, half - i
    J += np.bincount(i, weights=q * (1.0 - fr), minlength=n + 1)
    J += np.bincount(i + 1, weights=q * fr, minlength=n + 1)
    c = np.floor(xs)
    left, right = c < 2, c > n - 3
    x[on], u[on] = np.where(left, 1.5, np.where(right, n - 1.5, xs)), us
    alive[on[left | right]] = False
    return J


def _exact_step(s):
    """One Lorentz step of the reference's per-step functions on the prepared arrays."""
    V, P, C, st = s["V"], s["P"], s["C_V"], s["start"]
    N, W, f, r = P.Nz, P.pmlWidth, P.materialFrontEdge, P.materialRearEdge
    Ex, Hy, Dx, Pc, psE, psH = (st[k].copy() for k in ("Ex", "Hy", "Dx", "polarisationCurr", "psi_Ex", "psi_Hy"))
    g, dt, wp, w0 = V.gammaE, P.delT, V.plasmaFreqE, V.omega_0E
    den = 1.0 / dt ** 2 + g / (2.0 * dt)
    A, B = (2.0 / dt ** 2 - w0 ** 2) / den, (g / (2.0 * dt) - 1.0 / dt ** 2) / den
    Pc[f:r] = A * st["polarisationCurr"][f:r] + B * st["tempTempVarPol"][f:r] + P.permit_0 * wp ** 2 / den * Ex[f:r]
    Ex[1:N + 1] += (Hy[1:N + 1] - Hy[:N] - V.Jx[1:N + 1]) * V.UpExMat[1:N + 1] * C.den_Exdz[1:N + 1]
    for lo, hi in ((1, W), (N + 1 - W, N + 1)):
        psE[lo:hi] = C.beX[lo:hi] * psE[lo:hi] + C.ceX[lo:hi] * (Hy[lo:hi] - Hy[lo - 1:hi - 1])
        Ex[lo:hi] -= C.Cb[lo:hi] * psE[lo:hi]
    Dx[f:r] += dt / P.dz * (Hy[f:r] - Hy[f - 1:r - 1]) * C.den_Exdz[f:r]
    Ex[f:r] = (Dx[f:r] - Pc[f:r]) / P.permit_0
    Hy[1:N] = Hy[1:N] * V.UpHySelf[1:N] + (Ex[2:N + 1] - Ex[1:N]) * V.UpHyMat[1:N] * C.den_Hydz[1:N]
    for lo, hi in ((1, W), (N + 1 - W, N)):
        psH[lo:hi] = C.bmY[lo:hi] * psH[lo:hi] + C.cmY[lo:hi] * (Ex[lo + 1:hi + 1] - Ex[lo:hi])
        Hy[lo:hi] += C.C2[lo:hi] * psH[lo:hi]
    return dict(Ex=Ex, Hy=Hy, Dx=Dx, P=Pc, psi_Ex=psE, psi_Hy=psH)
