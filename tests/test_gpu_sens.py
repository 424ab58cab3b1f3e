"""cs_tran_sens (forward sensitivities of the plain-path transient) against
the reference's own answer and against the oracle.

- test/sensitivity.jl:13-44: the two-resistor divider, d out/dR1 = -d out/dR2
  = -out/2 at R1 = R2 = 1, at every output sample.
- Every other parameter kind against central differences of the oracle's
  transient at p +- h (h = 1e-6 |p|).  The sensitivities are those of the
  discrete solution on its step sequence, so the runs fix that sequence: with
  reltol = abstol = 1e6 every local error estimate is far below the growth
  cap, so each step doubles up to dt_max whatever p is (a tight tolerance
  lets an error estimate near the cap move the step times with p), and
  newton_tol 1e-15 on those weights converges Newton to about 1e-9.  A
  source's ".dc" is its value, DC and (for a DC source) transient alike, so
  its difference moves both.  Bar: 1e-6 of the parameter's largest
  sensitivity plus the differences' rounding floor.
"""
import numpy as np
import pytest

import cedarhip as ch
from cedarhip import lib as L
from cedarhip.netlist import WAVE_DC
from cedarhip.workloads import VDD, inverter, ring_oscillator
from oracle import oracle as O

import circuits as K

pytestmark = pytest.mark.gpu


# tolerances that keep the step sequence independent of the parameters
_FIXED = dict(reltol=1e6, abstol=1e6, newton_tol=1e-15)


def _say(msg):
    print(f"[gpu] {msg}", flush=True)


def test_divider_matches_reference(engine):
    _say("sens divider (test/sensitivity.jl)")
    flat = ch.lower(K.divider(1.0, 1.0))
    sys_ = engine.load(flat, solver=L.SOLVER_LEVEL)
    o = ch.grid_options((0.0, 1e-5), n_out=11)
    sol, sens = sys_.tran_sens(o, ["R1", "R2"])
    assert sol.retcode == "Success"
    out = sol["out"]
    q = sys_.probes.index(flat.index("out"))
    dR1, dR2 = sens[:, 0, q], sens[:, 1, q]
    np.testing.assert_allclose(dR1, -dR2, rtol=1e-12)
    np.testing.assert_allclose(dR1, -out / 2, rtol=1e-12)


def _indices(flat, nm):
    """The parameter vector entries a named sensitivity parameter moves."""
    idx = [flat.param_index(nm)]
    if nm.endswith(".dc"):
        kind, k = flat.device_names[nm.split(".")[0]]
        w = int(flat.arrays["vsrc_wave" if kind == "vsrc" else "isrc_wave"][k])
        if int(flat.arrays["wave_kind"][w]) == WAVE_DC:
            idx.append(flat.layout()["wave_data"] + int(flat.arrays["wave_off"][w]))
    return idx


def _fd_check(engine, flat, o, names, u0=None, rtol=1e-6):
    sys_ = engine.load(flat, solver=L.SOLVER_LEVEL)
    p = flat.params()
    sol, sens = sys_.tran_sens(o, names, u0=u0)
    assert sol.retcode == "Success", sol.retcode
    w0, _, st0, rc = O.tran(flat, p, u0, o)
    assert rc == 0 and st0.steps == sol.stats.steps
    for j, nm in enumerate(names):
        idx = _indices(flat, nm)
        h = 1e-6 * abs(p[idx[0]])
        pp, pm = p.copy(), p.copy()
        for i in idx:
            pp[i] += h
            pm[i] -= h
        wp, _, stp, rcp = O.tran(flat, pp, u0, o)
        wm, _, stm, rcm = O.tran(flat, pm, u0, o)
        assert rcp == 0 and rcm == 0
        assert stp.steps == st0.steps == stm.steps, (nm, stp.steps, st0.steps, stm.steps)
        fd = (wp - wm) / (2 * h)
        g = sens[:, j, :]
        # the largest sensitivity of this parameter, and the differences'
        # rounding floor (a few ulps of the waveform over 2h)
        bound = rtol * np.max(np.abs(fd)) + 100 * np.finfo(float).eps * np.max(np.abs(w0)) / h
        err = np.abs(g - fd)
        k, q = np.unravel_index(np.argmax(err - bound), err.shape)
        assert np.all(err <= bound), (nm, int(k), int(q), float(g[k, q]), float(fd[k, q]), bound)


def test_rc_ladder_and_source(engine):
    _say("sens RC/L/sources")
    flat = ch.lower(K.butterworth)
    o = ch.grid_options((0.0, 4.0), n_out=41, init=L.INIT_UIC, dt_max=0.01, **_FIXED)
    _fd_check(engine, flat, o, ["L1", "C2", "L3", "R4"], u0=np.zeros(flat.n))


def test_controlled_sources(engine):
    _say("sens controlled sources")
    flat = ch.lower(K.spice_controlled)
    o = ch.grid_options((0.0, 1e-6), n_out=5, dt_max=2e-8, **_FIXED)
    names = [nm for nm, (kind, k) in flat.device_names.items() if kind in ("vccs", "vcvs", "res")]
    names += [nm + ".dc" for nm, (kind, k) in flat.device_names.items() if kind in ("vsrc", "isrc")]
    _fd_check(engine, flat, o, names)


def test_inverter_mosfet_parameters(engine):
    """The inverter's PULSE transient from its DC point: MOSFET vth, kp, w,
    l, the load capacitance and the supply's DC value."""
    _say("sens inverter")
    flat = ch.lower(inverter())
    o = ch.grid_options((0.0, 2e-9), dt_out=20e-12, dt_max=1e-12, **_FIXED)
    _fd_check(engine, flat, o, ["MN.vth", "MN.kp", "MN.w", "MN.l", "MP.vth", "MP.w", "CL", "VDD.dc"])


def test_refuses_unsupported_parameters(engine):
    flat = ch.lower(inverter())
    sys_ = engine.load(flat, solver=L.SOLVER_LEVEL)
    lay = flat.layout()
    with pytest.raises(ch.CedarHIPError):
        sys_.tran_sens(ch.grid_options((0.0, 1e-10), n_out=3), [lay["gmin"]])


@pytest.mark.parametrize("case", ["inverter", "butterworth_uic", "controlled", "ring61_uic", "ring63_uic"])
def test_one_launch_matches_host_step_control(engine, case):
    """A sensitivity run of up to 64 unknowns goes in one launch; with
    BATCH_KERNEL_GLOBAL the host controls its steps.  The same rules on the
    same plan, with sums reduced over 64 lanes instead of 256: the same
    steps, and values equal up to rounding carried through the steps, held to
    the bar of the waveform parity tests (1e-6 relative) and 1e-9 of the
    parameter's largest sensitivity.  63 and 65 unknowns are the sizes beside the limit; the
    last takes the host's path either way."""
    u0, kw = None, {}
    if case == "inverter":
        flat, span = ch.lower(inverter()), (0.0, 1e-9)
        names = ["MN.vth", "MN.kp", "MP.w", "MP.l", "CL", "VDD.dc"]
    elif case == "butterworth_uic":
        flat, span = ch.lower(K.butterworth), (0.0, 4.0)
        names, u0 = ["L1", "C2", "L3", "R4"], np.zeros(flat.n)
    elif case == "controlled":
        flat, span = ch.lower(K.spice_controlled), (0.0, 1e-6)
        names = [nm for nm, (kind, k) in flat.device_names.items() if kind in ("vccs", "vcvs", "res")]
    else:
        ns = 61 if case == "ring61_uic" else 63
        flat, span = ch.lower(ring_oscillator(ns)), (0.0, 2e-11)
        names = ["MN0.vth", f"MP{ns - 1}.w", "VDD.dc"]
        u0 = np.zeros(flat.n)
        u0[flat.names["vdd"]] = VDD
        for k in range(ns):
            u0[flat.names[f"s{k}"]] = VDD * (k % 2)
    if u0 is not None:
        kw["init"] = L.INIT_UIC
    sys_ = engine.load(flat, solver=L.SOLVER_LEVEL)
    run = {}
    for kern in (L.BATCH_KERNEL_AUTO, L.BATCH_KERNEL_GLOBAL):
        o = ch.grid_options(span, n_out=21, batch_kernel=kern, **kw)
        run[kern] = sys_.tran_sens(o, names, flat.params(), u0=u0)
    (ra, ga), (rg, gg) = run[L.BATCH_KERNEL_AUTO], run[L.BATCH_KERNEL_GLOBAL]
    assert ra.retcode == rg.retcode == "Success"
    assert ra.stats.steps == rg.stats.steps and ra.stats.rejected == rg.stats.rejected
    assert np.all(np.abs(ra.wave - rg.wave) <= 1e-6 * np.abs(rg.wave) + 1e-9)
    for j in range(len(names)):
        a, b = ga[:, j], gg[:, j]
        _say(f"{case} {names[j]}: max |s| {np.max(np.abs(b)):.3e}, difference {np.max(np.abs(a - b)):.2e}")
        assert np.all(np.abs(a - b) <= 1e-6 * np.abs(b) + 1e-9 * np.max(np.abs(b)) + 1e-300), names[j]


@pytest.mark.parametrize("n_out,probes", [(65, None), (3001, None), (20001, ["out"])])
def test_one_launch_fine_output_grid(engine, n_out, probes):
    """More samples due at a step than unknowns are probed: the one launch
    writes them lanes over the samples; waveform and sensitivities as with
    host step control (the bars of test_one_launch_matches_host_step_control)."""
    flat = ch.lower(inverter())
    names = ["MN.vth", "MP.w", "CL"]
    sys_ = engine.load(flat)
    if probes:
        sys_.set_probes(probes)
    run = [sys_.tran_sens(ch.grid_options((0.0, 0.3e-9), n_out=n_out, batch_kernel=k), names)
           for k in (L.BATCH_KERNEL_AUTO, L.BATCH_KERNEL_GLOBAL)]
    (ra, ga), (rg, gg) = run
    assert ra.retcode == rg.retcode == "Success" and ra.stats.steps == rg.stats.steps
    assert np.all(np.abs(ra.wave - rg.wave) <= 1e-6 * np.abs(rg.wave) + 1e-9)
    for j in range(len(names)):
        a, b = ga[:, j], gg[:, j]
        assert np.all(np.abs(a - b) <= 1e-6 * np.abs(b) + 1e-9 * np.max(np.abs(b)) + 1e-300), names[j]


@pytest.mark.parametrize("n_out", [21, 3001])
def test_one_launch_does_not_depend_on_the_parameters_beside(engine, n_out):
    """A parameter's sensitivity, the waveform, the state and the statistics are
    the same bits whichever parameters run beside it, in any order: the first
    parameter's wavefront writes what is common to all."""
    flat = ch.lower(inverter())
    sys_ = engine.load(flat)
    names = ["MN.vth", "MN.kp", "MP.w", "MP.l", "CL", "VDD.dc"]
    o = ch.grid_options((0.0, 0.3e-9), n_out=n_out)
    ref, gref = sys_.tran_sens(o, names)
    assert ref.retcode == "Success"
    for order in ([5], [2, 0], [3, 1, 4, 0, 5, 2]):
        r, g = sys_.tran_sens(o, [names[k] for k in order])
        assert np.array_equal(r.wave, ref.wave) and np.array_equal(r.u_final, ref.u_final)
        assert r.stats.steps == ref.stats.steps and r.stats.newton_iters == ref.stats.newton_iters
        for q, k in enumerate(order):
            assert np.array_equal(g[:, q], gref[:, k]), names[k]
