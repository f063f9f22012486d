"""Resident field launches (fdtd_set_resident) against one launch per S steps.

A resident launch runs a whole fdtd_run with every tile's window in registers
and the tiles' edge cells handed over through a mailbox.  Tile widths, owned
ranges and (FP64) the block length differ from the one-block tiles', yet every
result must be the same bits: fields, slab state, CPML psi, probes, snapshots.
Sizes sit where a plan can go wrong: a grid of one tile, a last cell alone, odd
sizes, slabs of a few cells and slabs that reach into a CPML strip, sources
beside a slab, more probes than a tile captures, runs shorter than a block,
runs cut into pieces, several simulations of different lengths.  A launch whose
waits are bounded to one microsecond gives up and is run again: the results
stay the same.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("E", "H", "D", "P", "PM", "PSIE", "PSIH")


def _phys(N, steps, slab="kerr", F=None, R=None, **kw):
    from fdtd_pic_amd import configs, engine
    rng = np.random.default_rng(N)
    F = N // 2 if F is None else F
    R = min(F + N // 4, N - N // 6) if R is None else R
    p = configs.base(N, steps, slab_start=F, slab_stop=F if slab == "none" else R, src_cell=min(60, N // 4),
                     src_t0=4e-15, src_tau=1.5e-15, src_amp=1.8e8, probes=[N // 5 if N < 300 else 45, N - min(40, N // 6)],
                     pml_width=min(32, N // 8))
    if slab == "kerr":
        p.update(chi3=1e-19, eps_inf=rng.uniform(1, 3, max(R - F, 0)))
    p.update(kw)
    return engine.physical_spec(p)


def _dropin(kind, Nz=700, T=500, W=90, **kw):
    """A pass of a drop-in integrator (snapshots every 50 steps, TFSF)."""
    import Solver_Engine as SE
    from refcases import product_objects, small_setup
    setup = small_setup(Nz=Nz, T=T, W=W, F=kw.pop("F", 330), R=kw.pop("R", Nz - 1), nzsrc=150)
    flags = dict(SineCont=True, TFSF=True)
    flags.update({"linlor": dict(LorentzMed=True), "nl": dict(nonLinMed=True), "free": {}}[kind])
    V, P, C_V, C_P = product_objects(setup, 9e9, **flags)
    if kind == "nl":
        P.FreeSpace, P.Periods = False, 1000
    if kind == "free":
        P.epsRe = 2.25
    plan = {"linlor": SE.plan_linlor, "nl": SE.plan_nl, "free": SE.plan_free_space}[kind](
        V, P, C_V, C_P, int(0.7 * T), int(0.05 * T))
    return plan.passes[-1][0]


def _run(specs, prec, resident, cuts=(), tiling=None, wait_us=0):
    from fdtd_pic_amd import engine
    with engine.Context(prec) as c:
        if tiling:
            c.set_tiling(*tiling)
        c.set_resident(resident, wait_us)
        sims = [c.add(s) for s in specs]
        active = c.resident_active()
        for n in cuts:
            c.run(n)
        c.run_all()
        out = []
        for sim, s in zip(sims, specs):
            o = {f: sim.read(f) for f in FIELDS if f in ("E", "H", "PSIE", "PSIH") or s.R > s.F}
            o["probes"], o["progress"] = sim.probes(), sim.progress()
            if s.snap_rows:
                o["snap"] = sim.snapshots()
            out.append(o)
    return active, out


def _same(specs, prec, tag, **kw):
    print(f"resident {prec} {tag}", flush=True)
    taken = kw.pop("taken", True)
    on, a = _run(specs, prec, True, **kw)
    kw.pop("wait_us", None)
    off, b = _run(specs, prec, False, **kw)
    assert on == taken and not off
    for k, (x, y) in enumerate(zip(a, b)):
        assert np.abs(y["E"]).max() > 0
        for f in y:
            assert np.array_equal(x[f], y[f]), (tag, k, f)


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("N,slab,kw", [
    (40, "none", {}), (127, "linear", {}), (192, "kerr", {}), (193, "kerr", {}), (1000, "linear", {}),
    (4097, "kerr", {}), (4098, "kerr", dict(F=2000, R=2003)), (3001, "kerr", dict(F=1500, R=1501)),
    (2500, "linear", dict(F=1200, R=2490)), (2500, "kerr", dict(F=70, R=2400)),
    (9001, "kerr", dict(src_cell=4490)), (6000, "kerr", dict(probes=[3000, 3001, 3002, 3050, 3100, 700])),
    (25013, "linear", {}), (65536, "kerr", {}), (30000, "none", {})])
def test_resident_equals_launch_per_block(prec, N, slab, kw):
    # FP32 has no resident class for more than two probes in a tile
    _same([_phys(N, 411, slab, **kw)], prec, f"N={N} {slab} {kw}", taken=prec == "f64" or len(kw.get("probes", ())) < 3)


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("tiling", [(1, 24), (2, 16), (2, 48)])
def test_resident_at_set_tilings(prec, tiling):
    _same([_phys(5000, 301)], prec, f"tiling {tiling}", tiling=tiling)


@pytest.mark.parametrize("kind,kw", [("linlor", {}), ("nl", {}), ("free", {}), ("linlor", dict(Nz=2111, T=333, F=900)),
                                     ("free", dict(Nz=1500, F=700, R=1200))])
def test_resident_dropin_passes(kind, kw):
    spec = _dropin(kind, **kw)
    assert spec.snap_rows > 0 and spec.tfsf
    _same([spec], "f64", f"{kind} {kw}")


@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_resident_several_simulations_and_pieces(prec):
    specs = [_phys(3000, 500), _phys(800, 260, "none"), _phys(5001, 611), _phys(1200, 90, "linear", chi3=0.0)]
    _same(specs, prec, "four simulations", cuts=(96, 5, 192))


@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_resident_gives_up_and_runs_again(prec):
    """Waits bounded to 1 us: the launch gives up where a wait takes longer,
    whatever was done stays unseen, and its steps are run again."""
    _same([_phys(9000, 900), _phys(2000, 333, "none")], prec, "1 us waits", wait_us=1, cuts=(96, 192))


def test_resident_not_taken():
    from fdtd_pic_amd import engine
    with engine.Context("f64") as c:
        s = c.add(_phys(1000, 100))
        assert c.resident_active()
        s.set_energy(1, 8)
        assert not c.resident_active()


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("slab,tiling", [("kerr", None), ("linear", (2, 48)), ("none", (2, 16)), ("kerr", (1, 24))])
def test_more_tiles_than_the_device_holds(prec, slab, tiling):
    # one launch per block of steps with the resident plan's tiles: grids of one
    # or two tiles, ragged ones, different lengths, a run cut into pieces
    grids = [(65536, {}), (65003, {}), (40, {}), (61007, dict(F=70, R=20000)), (193, {}),
             (4097, dict(F=2000, R=2003))] + [(65536 - 977 * i, {}) for i in range(19)]
    specs = [_phys(n, 120 + k, "none" if n == 40 else slab, **(kw if slab != "none" else {}))
             for k, (n, kw) in enumerate(grids)]
    _same(specs, prec, f"blocks {slab} {tiling}", taken=False, cuts=(37, 1), tiling=tiling)


@pytest.mark.parametrize("slab", ["kerr", "linear"])
def test_resident_f32_long_runs(slab):
    """Roundings that a run meets once in some 1e8 cell-steps: an emulated
    vacuum cell beside the slab whose compensation is half a unit of its value
    in the last place, so that E is not D."""
    for n in (25013, 24007, 23011, 22003, 9001, 5003):
        F = n // 2
        _same([_phys(n, 24001, slab, F=F, R=F + 400 + n % 100, src_cell=100, probes=[60, n - 42],
                     **(dict(chi3=0.0) if slab == "linear" else {}))], "f32", f"long {slab} {n}")


@pytest.mark.parametrize("interval", [1, 7, 48, 2 ** 30, 2 ** 31 - 2, 2 ** 31 - 1])
def test_resident_snapshot_intervals(interval):
    # up to the largest interval the library takes: no row then but the first, which stays empty
    spec = _phys(2100, 301, "linear")
    spec.snap_interval, spec.snap_rows = interval, min(301 // interval + 1, 40)
    _same([spec], "f64", f"snapshots every {interval}", cuts=(5, 96))


def _probe_sims(N, tile):
    """Three probes in adjacent cells, and three a one-block tile apart, around
    two of the one-block tiles' boundaries."""
    at = [b + k for b in (900 // tile * tile, 900 // tile * tile + tile) for k in (-3, -2, -1, 0, 1)]
    sets = [[a, a + 1, a + 2] for a in at] + [[a, a + tile, a + 2 * tile] for a in at]
    return [_phys(N, 1601, "none" if i % 2 else "kerr", src_cell=860, probes=p) for i, p in enumerate(sets)]


@pytest.mark.parametrize("N", [5000, 40000])
@pytest.mark.parametrize("tiling", [None, (1, 24), (2, 48), (2, 16), (4, 48)])
def test_resident_f32_records_every_probe(tiling, N):
    """The resident tiles are cut elsewhere than the one-block tiles, and no
    FP32 tile of theirs records more than two probes."""
    K, S = tiling or (4, 32)
    for spec in _probe_sims(N, 64 * K - 2 * S):
        on, a = _run([spec], "f32", True, tiling=tiling)
        off, b = _run([spec], "f32", False, tiling=tiling)
        cells = [p[0] for p in spec.probes]
        for k, (x, y) in enumerate(zip(a[0]["probes"], b[0]["probes"])):
            same, seen = np.array_equal(x, y), np.abs(y).max() > 0
            assert same and seen, (tiling, on, cells, k)


@pytest.mark.parametrize("tiling", [(1, 24), (2, 48), (2, 16)])
def test_blocks_f32_record_every_probe(tiling):
    # (three probes in one of the one-block tiles would take the whole batch off the block launches)
    tile = 64 * tiling[0] - 2 * tiling[1]
    specs = [_phys(65536, 1601) for _ in range(12)]
    specs += [s for s in _probe_sims(40000, tile) if len({p[0] // tile for p in s.probes}) > 1]
    on, a = _run(specs, "f32", True, tiling=tiling)
    off, b = _run(specs, "f32", False, tiling=tiling)
    assert not on
    for spec, x, y in zip(specs, a, b):
        same = np.array_equal(x["probes"], y["probes"])
        assert same, (tiling, [p[0] for p in spec.probes])


@pytest.mark.parametrize("slab,tiling", [("kerr", None), ("linear", None), ("none", None), ("kerr", (2, 48)),
                                         ("kerr", (2, 16)), ("kerr", (1, 24))])
@pytest.mark.parametrize("interval", [1, 7, 13, 48, 50, 1000])
def test_resident_f32_snapshots(slab, tiling, interval):
    """A snapshot step cuts a block, and FP32 rounding depends on a step's place
    in its block and on the class that a one-block tile with snapshots runs."""
    specs = []
    for n, kw in ((5003, {}), (2100, {}), (25013, dict(src_cell=4000))):
        s = _phys(n, 611, slab, **kw)
        s.snap_interval, s.snap_rows = interval, min(611 // interval + 1, 40)
        specs.append(s)
    _same(specs, "f32", f"snapshots every {interval}, {slab} {tiling}", cuts=(5, 96), tiling=tiling)


@pytest.mark.parametrize("interval", [2000, 2001])
def test_resident_f32_snapshots_long(interval):
    for n in (25013, 24007, 23011, 9001, 5003):
        F = n // 2
        s = _phys(n, 24001, "kerr", F=F, R=F + 400 + n % 100, src_cell=100, probes=[60, n - 42])
        s.snap_interval, s.snap_rows = interval, 13
        _same([s], "f32", f"long, snapshots every {interval}, {n}")


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("nth", [1, 2, 3])
def test_resident_give_up_is_run_again(prec, nth):
    """A give-up forced from the host, in the first, a middle and the last of
    three launches: that one and those behind it are run again, once."""
    from fdtd_pic_amd import engine
    specs = [_phys(9000, 900), _phys(2000, 333, "none")]
    S = 16
    with engine.Context(prec) as c:
        c.set_tiling(2, S)
        sims = [c.add(s) for s in specs]
        assert c.resident_active() and c.resident_counts() == (0, 0, 0)
        c.resident_fail(nth)
        for n in (6 * S, 2 * S, 5 * S):
            c.run(n)
        assert c.resident_counts() == (3, 0, 3)
        got = [{f: s.read(f) for f in ("E", "H", "PSIE", "PSIH")} | {"probes": s.probes()} for s in sims]
        assert c.resident_counts() == (3, 4 - nth, 0)
    with engine.Context(prec) as c:
        c.set_tiling(2, S)
        c.set_resident(False)
        sims = [c.add(s) for s in specs]
        c.run(13 * S)
        for s, g in zip(sims, got):
            for f in g:
                assert np.array_equal(g[f], s.probes() if f == "probes" else s.read(f)), f


def test_resident_errors():
    from fdtd_pic_amd import _capi, engine
    with engine.Context("f64") as c:
        for on, wait in ((2, 0), (-1, 0), (1, -1), (1, 60000001)):
            with pytest.raises(_capi.FdtdError):
                _capi.check(c.lib.fdtd_set_resident(c.h, on, wait))
        with pytest.raises(_capi.FdtdError):
            c.resident_fail(-1)
        assert c.lib.fdtd_set_resident(None, 1, 0) and c.lib.fdtd_resident_fail(None, 1)
        assert c.lib.fdtd_resident_active(None, None) and c.lib.fdtd_resident_counts(None, None, None, None)
        assert c.lib.fdtd_resident_counts(c.h, None, None, None) == 0


def _beam_spec(N, steps):
    from fdtd_pic_amd import configs, engine
    rng = np.random.default_rng(N)
    spec = engine.physical_spec(configs.base(N, steps, slab_start=60, slab_stop=90, src_cell=200, probes=[150, N - 60],
                                             src_t0=5e-15, src_tau=2e-15, src_amp=1e6))
    return spec, engine.Beam(300 + rng.uniform(0.0, 80, 2000), rng.normal(0.0, 0.15, (2000, 3)), -configs.E_CHARGE,
                             configs.M_ELECTRON, 1e9, configs.DT, configs.DZ)


def _play(prec, resident, script, fail=0):
    """Runs the script's calls on one context: ("run", n), ("add", spec),
    ("beam", spec, beam), ("write", sim), ("reset", sim), ("tiling", K, S),
    ("halo", h), ("read",).  The state of every simulation at the end, and the
    launches run again."""
    from fdtd_pic_amd import engine
    with engine.Context(prec) as c:
        c.set_tiling(2, 16)
        c.set_resident(resident)
        if resident:
            c.resident_fail(fail)
        sims, out = [], []
        for what, *a in script + [("read",)]:
            if what == "run":
                c.run(a[0])
            elif what == "add":
                sims.append(c.add(a[0]))
            elif what == "beam":
                sims.append(c.add(a[0], beam=a[1]))
            elif what == "write":
                x = np.arange(sims[a[0]].spec.N + 1)
                sims[a[0]].write("E", 1e6 * np.exp(-((x - 300.0) / 40.0) ** 2))
            elif what == "reset":
                sims[a[0]].reset()
            elif what == "tiling":
                c.set_tiling(*a)
            elif what == "halo":
                c.set_halo_exchange(*a)
            else:
                for s in sims:
                    out.append({f: s.read(f) for f in ("E", "H", "PSIE", "PSIH") + (("D", "P") if s.spec.R > s.spec.F
                                                                                   else ())})
                    out[-1]["probes"], out[-1]["progress"] = s.probes(), s.progress()
                    if s.beam_n:
                        out[-1]["x"], out[-1]["u"], _ = s.particles()
        return out, c.resident_counts()[1]


def _plays_the_same(prec, script, fail=1, again=None):
    got, n = _play(prec, True, script, fail)
    want, _ = _play(prec, False, script)
    assert n > 0 if again is None else n == again
    for k, (x, y) in enumerate(zip(got, want)):
        assert np.abs(y["E"]).max() > 0 or y["progress"] == 0
        for f in y:
            same = np.array_equal(x[f], y[f])
            assert same, (k, f)


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("kind", ["add", "add and read", "write", "two", "beam", "beam, no run"])
def test_simulation_added_behind_a_launch_that_gives_up(prec, kind):
    """A simulation that is added while a resident launch is under way has no
    part in that launch's steps, also where they are run again."""
    a, b = ("add", _phys(5000, 500)), ("add", _phys(3000, 400, "none"))
    beam = ("beam", *_beam_spec(700, 200))
    run = ("run", 96)
    _plays_the_same(prec, {"add": [a, run, b, run], "add and read": [a, run, b, ("read",), run, ("read",), run],
                           "write": [a, run, b, ("write", 1), run, run],
                           "two": [a, run, b, ("add", _phys(801, 300)), run, run],
                           "beam": [a, run, beam, ("run", 32), ("read",), ("run", 7)],
                           "beam, no run": [a, run, beam]}[kind])


@pytest.mark.parametrize("change", [("tiling", 1, 24), ("tiling", 4, 32), ("tiling", 2, 32), ("halo", 8)])
def test_tiling_changed_behind_a_launch_that_gives_up(change):
    # FP32 rounding depends on the tiling: the steps before the change keep the old one
    a = ("add", _phys(5000, 500))
    _plays_the_same("f32", [a, ("run", 96), change, ("run", 96)])


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("cuts", [(101, 192), (69, 1, 192, 23), (96, 21, 17)])
def test_runs_keep_their_pieces_when_run_again(prec, cuts):
    """Several queued runs, none a whole number of blocks: FP32 rounding depends
    on where a block begins."""
    a, b = ("add", _phys(5000, 900)), ("add", _phys(3000, 400, "none"))
    _plays_the_same(prec, [a, b] + [("run", n) for n in cuts], again=len(cuts))


@pytest.mark.parametrize("tiling", [(2, 21), (4, 48)])
def test_resident_f32_very_long_run(tiling):
    # more steps than one launch takes: the cut falls between blocks
    spec = _phys(700, (1 << 20) + 300, "none", probes=[200])
    spec.srcE = 1e8 * np.sin(0.3 * np.arange(spec.steps))
    _same([spec], "f32", f"1,048,876 steps at {tiling}", tiling=tiling)


def test_busy_behind_a_give_up():
    # steps that are queued again are work: no "idle" before they have run
    from fdtd_pic_amd import engine
    with engine.Context("f64") as c:
        c.add(_phys(65536, 20000))
        c.resident_fail(1)
        c.run_all()
        seen = []
        while len(seen) < 200 or seen[-1]:
            seen.append(c.busy())
        assert True in seen and seen == sorted(seen, reverse=True)
        assert c.resident_counts() == (1, 1, 0)


def test_resident_pauses_after_a_give_up():
    """Something else holds the device: the runs after a give-up do not each
    wait for their bound again, until a second has passed."""
    import time
    from fdtd_pic_amd import engine
    with engine.Context("f64") as c:
        c.add(_phys(5000, 2000))
        c.resident_fail(1)
        for _ in range(5):
            c.run(100)
            c.sync()
        assert c.resident_counts() == (1, 1, 0) and not c.resident_active()
        time.sleep(1.1)
        assert c.resident_active()
        c.resident_fail(1)
        for _ in range(3):
            c.run(100)
            c.sync()
        time.sleep(1.1)                       # the second time it is two
        assert c.resident_counts() == (2, 2, 0) and not c.resident_active()
        time.sleep(1.0)
        for _ in range(3):
            c.run(100)
            c.sync()
        assert c.resident_counts() == (5, 2, 0)
        c.resident_fail(1)
        c.run(100)
        c.sync()
        assert not c.resident_active()
        c.set_resident(True)                  # asked for: at once
        assert c.resident_active()


@pytest.mark.parametrize("fail", [0, 1, 700, 2900])
def test_resident_queue_is_bounded(fail):
    """A loop of short runs: the host keeps track of so many launches only,
    and of the right ones when one of them gives up."""
    from fdtd_pic_amd import engine
    spec = _phys(2000, 300000)
    with engine.Context("f64") as c:
        s = c.add(spec)
        c.resident_fail(fail)
        most = 0
        for _ in range(3000):
            c.run(100)
            most = max(most, c.resident_counts()[2])
        got = {f: s.read(f) for f in ("E", "H", "D", "P")} | {"probes": s.probes()}
        assert s.progress() == 300000 and (c.resident_counts()[1] > 0) == (fail > 0)
    assert most <= 1024
    with engine.Context("f64") as c:
        c.set_resident(False)
        s = c.add(spec)
        c.run_all()
        for f in got:
            same = np.array_equal(got[f], s.probes() if f == "probes" else s.read(f))
            assert same, f


def test_reset_add_and_run_wait_for_nothing():
    from fdtd_pic_amd import engine
    with engine.Context("f64") as c:
        a = c.add(_phys(65536, 120000))
        b = c.add(_phys(2000, 120000, "none"))
        c.run(10)
        a.reset()
        b.reset()
        c.run(10)                             # the arrays that grow have grown
        c.sync()
        c.run(60000)
        a.reset()
        c.run(60000)
        c.add(_phys(1000, 2000))
        b.reset()
        c.run(100)
        assert c.resident_active() and c.resident_counts()[2] == 3 and c.busy()
        c.sync()
        assert c.resident_counts()[1:] == (0, 0)


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("fail", [1, 2, 3, 4])
@pytest.mark.parametrize("kind", ["reset", "all reset", "reset twice", "reset and add", "short", "blocks behind",
                                  "beam behind"])
def test_reset_and_add_between_runs_that_give_up(prec, fail, kind):
    """Each of several queued runs has other simulations, or the same ones begun
    anew: the ones that are run again have those that they had."""
    a, b, s = ("add", _phys(5000, 500)), ("add", _phys(3000, 400, "none")), ("add", _phys(801, 120))
    r = ("run", 64)
    script = {
        "reset": [a, b, r, ("reset", 0), r, r, ("reset", 1), ("run", 37)],
        "all reset": [a, b, r, ("reset", 0), ("reset", 1), ("run", 32), ("reset", 0), ("reset", 1), r, ("run", 5)],
        "reset twice": [a, b, r, ("reset", 0), ("reset", 0), r, ("reset", 0), r, ("run", 16)],
        "reset and add": [a, r, b, r, ("reset", 0), s, r, ("reset", 2), ("run", 70)],
        # simulations that end inside a run, before others begin
        "short": [s, ("run", 300), a, ("run", 300), ("reset", 0), ("run", 300), b, ("run", 450)],
        "blocks behind": [a, b, r, ("reset", 0), r, r, ("halo", 8), r, ("halo", 0), ("reset", 1), r],
        "beam behind": [a, b, r, ("reset", 0), r, r, ("beam", *_beam_spec(700, 200)), ("run", 33), ("read",), ("run", 9)],
    }[kind]
    _plays_the_same(prec, script, fail=fail, again=None if fail < 4 else 0 if kind == "beam behind" else 1)


@pytest.mark.parametrize("threads", [False, True])
def test_resident_contexts_share_the_device(threads):
    """A launch is taken while the tiles of all contexts' launches fit on the
    device together; the others run one block per launch.  Same bits."""
    from concurrent.futures import ThreadPoolExecutor
    from fdtd_pic_amd import engine
    big, small = _phys(65536, 30000), _phys(2000, 3000)
    with engine.Context("f64") as a, engine.Context("f64") as b, engine.Context("f32") as d, engine.Context("f64") as e:
        sims = [a.add(big), b.add(big), d.add(small), e.add(small)]
        for c in (a, b, d, e):
            assert c.resident_active()
        if threads:
            def go(c):
                for _ in range(30):
                    c.run(c is a and 1000 or 100)
                    c.sync()
            with ThreadPoolExecutor(4) as ex:
                list(ex.map(go, (a, b, d, e)))
            b.run(27000)
        else:
            a.run_all()
            assert a.busy()
            b.run(100)                        # while a's launch holds the device
            assert b.resident_counts()[0] == 0
            for c in (d, e):
                c.run(100)
            for c in (a, b, d, e):
                c.sync()
            b.run(100)                        # and after it
            d.run(2900)
            e.run(2900)
            b.run(29800)
            assert b.resident_counts()[0] > 0
        got = [{f: s.read(f) for f in ("E", "H", "D", "P")} | {"probes": s.probes()} for s in sims]
    for k, (prec, spec) in enumerate((("f64", big), ("f64", big), ("f32", small), ("f64", small))):
        if k == 1:
            continue
        with engine.Context(prec) as c:
            c.set_resident(False)
            s = c.add(spec)
            if prec == "f32" and threads:
                for _ in range(30):
                    c.run(100)
            elif prec == "f32":
                c.run(100)
            c.run_all()
            for f in got[k]:
                want = s.probes() if f == "probes" else s.read(f)
                same = np.array_equal(got[k][f], want) and (k > 0 or np.array_equal(got[1][f], want))
                assert same, (k, f)


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("tiling", [None, (2, 16), (4, 48), (1, 24)])
@pytest.mark.parametrize("fail", [0, 1])
def test_runs_of_one_block(prec, tiling, fail):
    """Runs that end within a block, alone and behind resident launches, one
    of which gives up."""
    a, b = _phys(5000, 900), _phys(3000, 400, "none")
    b.snap_interval, b.snap_rows = 7, 40
    script = [("tiling", *tiling)] if tiling else []
    script += [("add", a), ("add", b)] + [("run", n) for n in (1, 1, 5, 16, 150, 1, 3, 24, 110)] + [("read",)]
    script += [("run", n) for n in (7, 2)] + [("reset", 0), ("run", 9), ("read",), ("run", 130), ("run", 4)]
    _plays_the_same(prec, script, fail=fail, again=None if fail else 0)


def test_short_runs_are_no_resident_launches():
    from fdtd_pic_amd import engine
    for prec in ("f32", "f64"):
        with engine.Context(prec) as c:
            c.add(_phys(5000, 2000))
            assert c.resident_active()
            for _ in range(20):
                c.run(1)
                c.run(16)
            assert c.resident_counts() == (0, 0, 0)
            c.run(500)
            assert c.resident_counts() == (1, 0, 1)


@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_simulation_removed_behind_a_launch_that_gives_up(prec):
    from fdtd_pic_amd import engine
    specs = [_phys(5000, 900), _phys(3000, 400, "none"), _phys(801, 300)]
    out = []
    for resident in (True, False):
        with engine.Context(prec) as c:
            c.set_tiling(2, 16)
            c.set_resident(resident)
            c.resident_fail(2 if resident else 0)
            sims = [c.add(s) for s in specs[:2]]
            c.run(96)
            c.run(64)
            sims[0].remove()
            assert c.resident_counts()[1] == (1 if resident else 0)
            sims.append(c.add(specs[2]))
            c.run(80)
            out.append([s.read(f) for s in sims[1:] for f in ("E", "H", "PSIE")] + [s.probes() for s in sims[1:]])
    for x, y in zip(*out):
        assert np.array_equal(x, y)
