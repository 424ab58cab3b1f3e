"""The packed launch's shapes against the oracle: instances per workgroup (one
for a batch below the CU count, up to eight), the two register budgets (a
batch past eight instances per CU takes the one for sixteen wavefronts), DC
and driven sources, one, two and four rows per lane, and circuits whose solve
has long tasks and updated diagonals (an RC mesh).  The step sequences are
equal, so waveforms agree to reltol 1e-6 / abstol 1e-9 V as in the other
parity tests."""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import cedarhip as ch
from cedarhip import lib as L
from cedarhip.engine import pack_plan
from cedarhip.workloads import NMOS, PMOS, VDD, inverter, rc_mesh, ring_initial_state, ring_oscillator
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _instances(kind, count, rng):
    flats, params, u0s = [], [], []
    made = {}
    for i in range(count):
        if kind == "rings":
            n = (5, 33, 67)[i % 3]
            f = made.setdefault(n, ch.lower(ring_oscillator(n)))
        elif kind == "inverters":
            f = made.setdefault(0, ch.lower(inverter()))
        elif kind == "wide":
            f = made.setdefault(0, ch.lower(ring_oscillator(149)))
        else:
            f = made.setdefault(0, rc_mesh(7, 6, 5, seed=3))
        p = f.params()
        lay = f.layout()
        nm = len(f.arrays["mos_vth"])
        p[lay["mos_vth"]:lay["mos_vth"] + nm] += 0.03 * rng.standard_normal(nm)
        flats.append(f)
        params.append(p)
        u0s.append(ring_initial_state(f, rng) if kind in ("rings", "wide") else None)
    return flats, params, (u0s if kind in ("rings", "wide") else None)


@pytest.mark.parametrize("kind,count", [("rings", 7), ("rings", 259), ("rings", 2051), ("inverters", 3),
                                        ("inverters", 1030), ("inverters", 2051), ("wide", 5), ("wide", 300),
                                        ("mesh", 2), ("mesh", 2051)])
def test_packed_shapes_match_oracle(engine, kind, count):
    print(f"[gpu] packed shapes {kind} {count}", flush=True)
    rng = np.random.default_rng(count)
    flats, params, u0s = _instances(kind, count, rng)
    span = {"rings": 8e-12, "inverters": 0.25e-9, "wide": 2e-12, "mesh": 20e-12}[kind]
    o = ch.grid_options((0.0, span), n_out=5, init=L.INIT_UIC if u0s else L.INIT_DCOP,
                        batch_kernel=L.BATCH_KERNEL_LDS)
    r = ch.tran_batch(flats, params, o, u0=u0s, engine=engine)
    assert set(r.retcodes) == {"Success"}
    pick = sorted({0, 1, count // 2, count - 2, count - 1} & set(range(count)))
    w, uf, st, rc = O.tran_batch([flats[i] for i in pick], [params[i] for i in pick],
                                 [u0s[i] for i in pick] if u0s else None, o)
    assert rc == 0
    for q, i in enumerate(pick):
        assert r.stats[i].steps == st[q].steps
        assert np.all(np.abs(r.wave[i] - w[q]) <= 1e-6 * np.abs(w[q]) + 1e-9)
        assert np.all(np.abs(r.u_final[i] - uf[q]) <= 1e-6 * np.abs(uf[q]) + 1e-9)


@pytest.mark.parametrize("name", ["inverter", "ring5", "ring67", "ring149", "mesh", "butterworth", "vr"])
def test_cs_tran_and_dcop_take_one_launch(engine, name):
    """cs_tran and cs_dcop by default, on the LDS-resident kernel, against the
    plain path (batch_kernel = CS_BATCH_KERNEL_GLOBAL) and the oracle, with
    probes, without an output grid, and a second call with other values."""
    import circuits as K
    print(f"[gpu] single launch {name}", flush=True)
    rng = np.random.default_rng(4)
    u0 = None
    if name.startswith("ring"):
        flat, span = ch.lower(ring_oscillator(int(name[4:]))), 4e-12
        u0 = ring_initial_state(flat, rng)
    else:
        flat, span = {"inverter": (ch.lower(inverter()), 0.3e-9), "mesh": (rc_mesh(7, 6, 5, seed=3), 20e-12),
                      "butterworth": (ch.lower(K.butterworth), 0.5), "vr": (ch.lower(K.vr), 1e-3)}[name]
    s = engine.load(flat, solver=L.SOLVER_LEVEL)
    kw = {"init": L.INIT_UIC} if u0 is not None else {}
    for trial in range(2):
        p = flat.params()
        if trial and len(flat.arrays["mos_vth"]):
            p[flat.layout()["mos_vth"]] += 0.05
        o = ch.grid_options((0.0, span), n_out=7, **kw)
        w, uf, st, rc = O.tran(flat, p, u0, o)
        a = s.tran(o, p, u0)
        b = s.tran(ch.grid_options((0.0, span), n_out=7, batch_kernel=L.BATCH_KERNEL_GLOBAL, **kw), p, u0)
        c = s.tran(ch.TranOptions(t_start=0.0, t_stop=span, **kw), p, u0)
        assert a.retcode == b.retcode == c.retcode == "Success" and rc == 0
        assert a.stats.steps == b.stats.steps == st.steps and a.stats.newton_iters == b.stats.newton_iters
        for r in (a, b):
            assert np.all(np.abs(r.wave - w) <= 1e-6 * np.abs(w) + 1e-9)
            assert np.all(np.abs(r.u_final - uf) <= 1e-6 * np.abs(uf) + 1e-9)
        assert np.array_equal(c.u_final, a.u_final) and c.wave.shape[0] == 0
        if u0 is None:
            ud, _, rcd = O.dcop(flat, p)
            for dc in (s.dcop(p), s.dcop(p, ch.TranOptions(batch_kernel=L.BATCH_KERNEL_GLOBAL))):
                assert dc.retcode == "Success" and rcd == 0
                assert np.max(np.abs(dc.u - ud)) <= 1e-9 * max(1.0, np.max(np.abs(ud)))
    s.set_probes([1, 0])
    d = s.tran(ch.grid_options((0.0, span), n_out=7, **kw), p, u0)
    assert np.array_equal(d.wave, a.wave[:, [1, 0]])


def test_early_stop_leaves_later_samples(engine):
    """A run that ends at max_steps fills the samples up to its time only, on both kernels."""
    print("[gpu] early stop", flush=True)
    flat = ch.lower(inverter())
    s = engine.load(flat)
    for kern in (L.BATCH_KERNEL_AUTO, L.BATCH_KERNEL_GLOBAL):
        r = s.tran(ch.grid_options((0.0, 1e-9), n_out=101, max_steps=150, batch_kernel=kern))
        assert r.retcode == "MaxIters" and r.stats.steps + r.stats.rejected == 150
        done = r.t <= r.stats.t_end * (1 + 1e-9)
        assert done.any() and not done.all()
        assert np.all(r.wave[done, 0] > 1.0) and np.all(r.wave[~done] == 0.0)


@pytest.mark.parametrize("kern,m", [(L.BATCH_KERNEL_AUTO, 83_886), (L.BATCH_KERNEL_AUTO, 83_887),
                                    (L.BATCH_KERNEL_AUTO, 100_000), (L.BATCH_KERNEL_LDS, 100_000),
                                    (L.BATCH_KERNEL_LDS, 130_000)])
def test_large_sample_buffer_is_given_back(engine, kern, m):
    """64 MiB of samples, the most that AUTO takes on the one launch, and more:
    on the plain path, and on the one launch when asked for, whose buffer is
    kept or freed after the call.  The next calls, large and small, give the
    same samples (every m-th sample of the large run is one of the small
    run's)."""
    print(f"[gpu] large sample buffer, kernel {kern}, 20 x {m}", flush=True)
    flat = ch.lower(inverter())
    s = engine.load(flat)
    n_out = 20 * m + 1
    assert (n_out * len(s.probes) * 8 > 64 << 20) == (m > 83_886)
    runs = [s.tran(ch.grid_options((0.0, 1e-9), n_out=k, batch_kernel=kern)) for k in (21, n_out, 21, n_out)]
    assert all(r.retcode == "Success" for r in runs)
    assert np.array_equal(runs[0].wave, runs[2].wave) and np.array_equal(runs[1].wave, runs[3].wave)
    assert np.all(np.abs(runs[1].wave[::m] - runs[0].wave) <= 1e-9 * np.abs(runs[0].wave) + 1e-9)


def _free_device_memory():
    hip = ctypes.CDLL("libamdhip64.so.7")   # the runtime the library itself links
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_sample_buffers_do_not_add_up_over_circuits():
    """Twelve circuits of one context, each run with 30 MiB of samples: the
    context keeps one buffer for all of them (each had kept its own, and as
    much pinned host memory)."""
    print("[gpu] sample buffers over circuits", flush=True)
    eng = ch.Engine(0)
    try:
        flat = ch.lower(inverter())
        systems = [eng.load(flat) for _ in range(12)]
        n_out = (30 << 20) // (8 * len(systems[0].probes))
        free = []
        for s in systems:
            assert s.tran(ch.grid_options((0.0, 1e-10), n_out=n_out)).retcode == "Success"
            free.append(_free_device_memory())
        assert free[0] - free[-1] <= 16 << 20
    finally:
        eng.close()


@pytest.mark.parametrize("kern", [L.BATCH_KERNEL_AUTO, L.BATCH_KERNEL_LDS])
def test_two_threads_on_one_context(engine, kern):
    """Two threads, each with a circuit of its own in the same context: every
    run gives the samples it gives alone."""
    print(f"[gpu] two threads, kernel {kern}", flush=True)
    systems = [engine.load(ch.lower(inverter())), engine.load(ch.lower(inverter(cload=25e-15)))]
    opts = [ch.grid_options((0.0, 3e-10), n_out=k, batch_kernel=kern) for k in (31, 60_001)]
    alone = [[s.tran(o).wave for o in opts] for s in systems]
    with ThreadPoolExecutor(2) as ex:
        got = list(ex.map(lambda s: [s.tran(opts[q % 2]).wave for q in range(12)], systems))
    for g, a in zip(got, alone):
        assert all(np.array_equal(w, a[q % 2]) for q, w in enumerate(g))


def test_infinite_tolerance_and_span(engine):
    """abstol = inf weighs every error with 0: each step converges in one
    iteration and is accepted.  An infinite t_stop has no default for dt_max,
    and the run ends at max_steps.  The LDS-resident kernels divide by a
    reciprocal of their own, so 1/inf and inf/x are theirs to get right: the
    one launch and a batch take the plain path's and the oracle's steps."""
    print("[gpu] infinite abstol, infinite t_stop", flush=True)
    flat = ch.lower(inverter())
    s = engine.load(flat)
    p = flat.params()
    for kw, n_out, want in (({"abstol": np.inf, "t_stop": 1e-9, "dt_out": 2.5e-10}, 5, "Success"),
                            ({"t_stop": np.inf, "dt_init": 1e-13, "dt_min": 1e-20, "max_steps": 60}, 0, "MaxIters")):
        runs = []
        for kern in (L.BATCH_KERNEL_AUTO, L.BATCH_KERNEL_GLOBAL):
            r = s.tran(ch.TranOptions(n_out=n_out, batch_kernel=kern, **kw), p)
            runs.append((r.retcode, r.stats, r.wave, r.u_final))
        o = ch.TranOptions(n_out=n_out, batch_kernel=L.BATCH_KERNEL_LDS, **kw)
        b = ch.tran_batch([flat, flat], [p, p], o, engine=engine)
        runs += [(b.retcodes[i], b.stats[i], b.wave[i], b.u_final[i]) for i in range(2)]
        w, uf, st, rc = O.tran(flat, p, None, o)
        for code, stats, wave, u in runs:
            assert code == want
            assert (stats.steps, stats.rejected, stats.newton_iters) == (st.steps, st.rejected, st.newton_iters)
            assert np.all(np.abs(wave - w[:n_out]) <= 1e-6 * np.abs(w[:n_out]) + 1e-9)
            assert np.all(np.abs(u - uf) <= 1e-6 * np.abs(uf) + 1e-9)


def test_dcop_kernel_choice(engine):
    """cs_dcop runs on the kernel that batch_kernel names.  Without charges the
    initial point of a transient is the DC point itself, so a run of no steps
    returns each kernel's own point, to the bit; the two kernels sum in
    another order, and over a few parameter sets their points differ."""
    print("[gpu] dcop kernel choice", flush=True)

    def circuit():
        vdd, vin, gnd = (ch.Named(ch.net, k)() for k in ("vdd", "in", "gnd"))
        ch.Named(ch.V(VDD), "VDD")(vdd, gnd)
        ch.Named(ch.V(0.85), "VIN")(vin, gnd)
        a = vin
        for k in range(8):
            y = ch.Named(ch.net, f"s{k}")()
            ch.Named(ch.SquareLawMOSFET(**NMOS), f"MN{k}")(y, a, gnd, gnd)
            ch.Named(ch.SquareLawMOSFET(**PMOS), f"MP{k}")(y, a, vdd, vdd)
            a = y
        ch.Gnd()(gnd)

    flat = ch.lower(circuit)
    s = engine.load(flat)
    lay = flat.layout()
    rng = np.random.default_rng(11)
    differ = 0
    for _ in range(8):
        p = flat.params()
        p[lay["mos_vth"]:lay["mos_vth"] + 16] += 0.02 * rng.standard_normal(16)
        ud, _, rcd = O.dcop(flat, p)
        u = {}
        for kern in (L.BATCH_KERNEL_AUTO, L.BATCH_KERNEL_GLOBAL):
            o = ch.TranOptions(t_stop=1e-9, max_steps=0, batch_kernel=kern)
            dc = s.dcop(p, o)
            assert dc.retcode == "Success" and rcd == 0
            assert np.max(np.abs(dc.u - ud)) <= 1e-9 * np.max(np.abs(ud))
            assert np.array_equal(dc.u, s.tran(o, p).u_final)
            u[kern] = dc.u
        differ += not np.array_equal(u[L.BATCH_KERNEL_AUTO], u[L.BATCH_KERNEL_GLOBAL])
    assert differ > 0


@pytest.mark.parametrize("n,count", [(101, 1300), (101, 2048), (149, 1536), (175, 1024)])
def test_lds_bound_batch_is_resident_at_once(engine, n, count):
    """Batches whose chunks hold five, three or two instances for LDS: two
    workgroups share a CU, so the launch lasts as long as its longest
    instance.  In two rounds it takes twice that."""
    print(f"[gpu] resident batch {n} {count}", flush=True)
    rng = np.random.default_rng(n)
    flat = ch.lower(ring_oscillator(n))
    u0 = ring_initial_state(flat, rng)
    chunks, _ = pack_plan([flat], [count])
    assert 256 < len(chunks) <= 512   # more than the CUs, no more than two each
    o = ch.TranOptions(t_stop=5e-12, init=L.INIT_UIC, batch_kernel=L.BATCH_KERNEL_LDS)
    s = engine.load(flat)
    b = ch.Batch(engine, [s], [0] * count, [flat.params()] * count, o, [u0] * count)
    try:
        b.run()
        ms = b.run()
        r = b.results(ms)
    finally:
        b.close()
    assert set(r.retcodes) == {"Success"}
    assert ms <= 1.4e3 * max(st.busy_s for st in r.stats)


@pytest.mark.parametrize("name,n_out,probes", [
    ("inverter", 2, None), ("inverter", 65, None), ("inverter", 5001, None), ("inverter", 20001, ["out"]),
    ("inverter", 3001, ["out", "VIN.I", "in"]), ("ring67", 4001, None), ("ring67", 30001, ["s66", "vdd", "s3", "s64"]),
    ("ring149", 3001, ["s148", "s0", "s70"])])
def test_fine_output_grids(engine, name, n_out, probes):
    """Output grids finer than the steps: up to hundreds of samples are due at
    one accepted point, written 64 at a time, lanes over the samples where
    more are due than rows are probed and over the rows otherwise.  cs_tran
    (AUTO and GLOBAL) and batches on both kernels against the oracle."""
    print(f"[gpu] fine grid {name} {n_out} {probes}", flush=True)
    rng = np.random.default_rng(n_out)
    u0 = None
    if name == "inverter":
        flat, span = ch.lower(inverter()), 0.3e-9
    else:
        flat, span = ch.lower(ring_oscillator(int(name[4:]))), 2e-12
        u0 = ring_initial_state(flat, rng)
    kw = {"init": L.INIT_UIC} if u0 is not None else {}
    p = flat.params()
    w, _, st, rc = O.tran(flat, p, u0, ch.grid_options((0.0, span), n_out=n_out, **kw))
    assert rc == 0
    s = engine.load(flat, solver=L.SOLVER_LEVEL)
    if probes:
        s.set_probes(probes)
        w = w[:, s.probes]
    runs = []
    for kern in (L.BATCH_KERNEL_AUTO, L.BATCH_KERNEL_GLOBAL, L.BATCH_KERNEL_LDS):
        o = ch.grid_options((0.0, span), n_out=n_out, batch_kernel=kern, **kw)
        r = s.tran(o, p, u0)
        assert r.retcode == "Success" and r.stats.steps == st.steps
        runs.append(r.wave)
        if kern != L.BATCH_KERNEL_AUTO:
            b = ch.Batch(engine, [s], [0, 0], [p, p], o, None if u0 is None else [u0, u0])
            try:
                b.run()
                runs += b.results().wave
            finally:
                b.close()
    for x in runs:
        assert np.all(np.abs(x - w) <= 1e-6 * np.abs(w) + 1e-9)


def test_samples_cost_less_than_the_run(engine):
    """200,001 samples of an inverter's run do not double its time on the
    device (one after the other they took ten times the run)."""
    print("[gpu] cost of samples", flush=True)
    s = engine.load(ch.lower(inverter()))
    busy = {}
    for n_out in (21, 200_001):
        for _ in range(2):
            r = s.tran(ch.grid_options((0.0, 1e-9), n_out=n_out, batch_kernel=L.BATCH_KERNEL_LDS))
        assert r.retcode == "Success"
        busy[n_out] = r.stats.busy_s
    print(f"[gpu] busy {busy}", flush=True)
    assert busy[200_001] <= 2.0 * busy[21]


def test_global_kernel_fills_the_device(engine):
    """4096 instances of a small circuit on the global-plan kernel are resident
    at once: they take a quarter longer than 2048, for the fuller CUs, and not
    twice as long."""
    print("[gpu] residency of the global-plan kernel", flush=True)
    flat = ch.lower(ring_oscillator(33))
    u0 = ring_initial_state(flat, np.random.default_rng(7))
    s = engine.load(flat)
    ms = {}
    for count in (2048, 4096):
        b = ch.Batch(engine, [s], [0] * count, [flat.params()] * count,
                     ch.TranOptions(t_stop=2e-12, init=L.INIT_UIC, batch_kernel=L.BATCH_KERNEL_GLOBAL), [u0] * count)
        try:
            ms[count] = min(b.run() for _ in range(3))
            assert set(b.results().retcodes) == {"Success"}
        finally:
            b.close()
    print(f"[gpu] kernel ms {ms}", flush=True)
    assert ms[4096] <= 1.5 * ms[2048]


@pytest.mark.parametrize("wave", ["damped_sine", "late_sine", "one_shot_pulse", "slow_pulse", "sine_cycles"])
def test_waveforms_on_every_kernel(engine, wave):
    """Sources whose values the batched and one-launch kernels compute by
    wave_math.h (damped and phase-shifted sines, a delayed one, one that ends
    after its cycles, a pulse with no period, one with a period the run passes
    twice) against the plain path, which calls the library, and the oracle."""
    from cedarhip.netlist import WAVE_PULSE, WAVE_SIN, Waveform
    print(f"[gpu] waveform {wave}", flush=True)
    w = {"damped_sine": (WAVE_SIN, [0.3, 1.2, 2.5e9, 1e-10, 1.5e9, 40.0, 1e30]),
         "late_sine": (WAVE_SIN, [0.9, -0.7, 1e9, 7e-10, 0.0, -75.0, 1e30]),
         "sine_cycles": (WAVE_SIN, [0.9, 0.8, 3e9, 0.0, 0.0, 200.0, 2.0]),
         "one_shot_pulse": (WAVE_PULSE, [0.1, 1.7, 2e-10, 5e-11, 8e-11, 3e-10, np.inf]),
         "slow_pulse": (WAVE_PULSE, [1.7, 0.1, 1e-10, 5e-11, 8e-11, 2e-10, 6e-10])}[wave]

    def circuit():
        vin, out, gnd = (ch.Named(ch.net, k)() for k in ("in", "out", "gnd"))
        ch.Named(ch.VoltageSource(tran=Waveform(*w)), "VIN")(vin, gnd)
        ch.Named(ch.R(1e3), "R")(vin, out)
        ch.Named(ch.C(1e-13), "C")(out, gnd)
        ch.Gnd()(gnd)

    flat = ch.lower(circuit)
    p = flat.params()
    s = engine.load(flat)
    ref, _, st, rc = O.tran(flat, p, None, ch.grid_options((0.0, 1.5e-9), n_out=61))
    assert rc == 0
    waves = []
    for kern in (L.BATCH_KERNEL_AUTO, L.BATCH_KERNEL_GLOBAL):
        o = ch.grid_options((0.0, 1.5e-9), n_out=61, batch_kernel=kern)
        r = s.tran(o, p)
        assert r.retcode == "Success" and r.stats.steps == st.steps
        waves.append(r.wave)
        b = ch.tran_batch([flat] * 2, [p, p], o, engine=engine)
        assert b.retcodes == ["Success"] * 2 and b.stats[1].steps == st.steps
        waves += b.wave
        waves.append(s.tran_sens(o, ["R"], p)[0].wave)
    for x in waves:
        assert np.all(np.abs(x - ref) <= 1e-6 * np.abs(ref) + 1e-9)
