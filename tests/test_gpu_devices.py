"""GPU parity of every linear device, source waveform and m-factor, on the
reference's own test circuits (tests/circuits.py).

Each circuit runs through the plain path (cs_residual / cs_jacobian, cs_dcop,
cs_tran) and through both batched kernels (all the circuits in one launch, so
the batch is uneven), and is compared with the oracle (stamps 1e-12 relative;
waveforms reltol 1e-6 / abstol 1e-9 with identical accepted-step counts) and
with the answers the reference's tests assert.
"""
import json
import os

import numpy as np
import pytest

import cedarhip as ch
from cedarhip import lib as L
from oracle import oracle as O

import circuits as K

pytestmark = pytest.mark.gpu

GOLD = json.load(open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden",
                                   "reference_answers.json")))


def _say(msg):
    print(f"[gpu] {msg}", flush=True)


def _close(a, b, rtol, atol):
    a, b = np.asarray(a), np.asarray(b)
    return np.all(np.abs(a - b) <= rtol * np.maximum(np.abs(a), np.abs(b)) + atol)


DC_CIRCUITS = [("vr", K.vr), ("ir", K.ir), ("spice_controlled", K.spice_controlled),
               ("multiplicities", K.multiplicities), ("divider", K.divider(300.0, 1700.0)),
               ("butterworth", K.butterworth), ("multi_vrc", K.multi_vrc)]


@pytest.mark.parametrize("name,fn", DC_CIRCUITS)
@pytest.mark.parametrize("solver", [L.SOLVER_LEVEL, L.SOLVER_SUPERNODAL])
def test_residual_jacobian_linear_devices(engine, name, fn, solver):
    """f!/jac! of inductors, controlled sources, PWL/SIN sources and m-factors
    against the oracle at 1e-12, on the level-scheduled and supernodal paths."""
    _say(f"residual/jacobian {name} solver {solver}")
    flat = ch.lower(fn)
    sys = engine.load(flat, solver=solver)
    p = flat.params()
    rng = np.random.default_rng(11)
    for _ in range(3):
        u = rng.uniform(-2.0, 2.0, flat.n)
        du = 1e3 * rng.standard_normal(flat.n)
        for t, mode in ((0.37, L.MODE_TRAN), (0.0, L.MODE_DCOP)):
            r_gpu = sys.f(None, du, u, p, t, mode)
            r_ref = O.residual(flat, p, u, du, t, mode)
            assert np.max(np.abs(r_gpu - r_ref)) <= 1e-12 * (np.max(np.abs(r_ref)) + 1e-30), (name, mode)
            J_gpu = sys.jac_matrix(du, u, p, 2.5e3, t, mode).toarray()
            J_ref = O.jacobian(flat, p, u, 2.5e3, t, mode)
            assert np.max(np.abs(J_gpu - J_ref)) <= 1e-12 * np.max(np.abs(J_ref)), (name, mode)


@pytest.mark.parametrize("name,fn", DC_CIRCUITS[:5])
def test_dcop_reference_answers(engine, name, fn):
    """dc! on the GPU: the oracle's solution and the reference's answers."""
    _say(f"dcop {name}")
    flat = ch.lower(fn)
    sol = engine.load(flat).dcop()
    u_ref, _, rc = O.dcop(flat, flat.params())
    assert sol.retcode == "Success" and rc == 0
    assert _close(sol.u, u_ref, 1e-12, 1e-15)
    if name == "vr":
        assert sol["V.I"] == pytest.approx(GOLD["simple_vr"]["i_source"], rel=1e-12)
    elif name == "ir":
        assert sol["icc"] == pytest.approx(GOLD["simple_ir"]["v_icc"], rel=1e-12)
    elif name == "spice_controlled":
        for k in ("node_5", "node_6", "node_7", "node_8", "node_9"):
            assert sol[k] == pytest.approx(GOLD["spice_controlled"][k], rel=1e-12)
    elif name == "multiplicities":
        for k in range(1, 7):
            assert sol[f"node_{k}"] == pytest.approx(10 / 11, rel=4e-16)
    elif name == "divider":
        assert sol["V.I"] == pytest.approx(-1 / 2000.0, rel=1e-12)


# (name, circuit, tspan, n_out, u0 or None (DC op), tolerances)
TRAN_CASES = [
    ("vrc", K.vrc, (0.0, 20e-3), 201, np.array([5.0, 0.0, 0.0]), 1e-8),
    ("multi_vrc", K.multi_vrc, (0.0, 2e-3), 201, np.array([5.0, 0.0, 0.0]), 1e-8),
    ("spectre_sources", K.spectre_sources, (0.0, 1.0), 11, None, 1e-8),
    ("pwl_current", K.pwl_current, (0.0, 10e-3), 201, None, 1e-8),
    ("butterworth", K.butterworth, (0.0, 30.0), 301, "zeros", 1e-10),
]


def _tran_case(case):
    name, fn, tspan, n_out, u0, tol = case
    flat = ch.lower(fn)
    if isinstance(u0, str):
        u0 = np.zeros(flat.n)
    init = L.INIT_UIC if u0 is not None else L.INIT_DCOP
    o = ch.grid_options(tspan, n_out=n_out, reltol=tol, abstol=tol, init=init)
    return name, flat, o, u0


def _check_reference(name, flat, o, w):
    t = o.t_start + o.dt_out * np.arange(o.n_out)
    if name == "vrc":
        assert w[0, flat.index("V.I")] == pytest.approx(GOLD["vrc"]["i_source_start"], rel=1e-12)
        assert np.max(np.abs(w[:, flat.index("vrc")] - 5.0 * (1 - np.exp(-t / 2e-3)))) < 5e-5
    elif name == "multi_vrc":
        assert w[0, flat.index("V.I")] == pytest.approx(-10 * 5.0 / 2000.0, rel=1e-12)
        assert np.max(np.abs(w[:, flat.index("vrc")] - 5.0 * (1 - np.exp(-t / 2e-4)))) < 5e-5
    elif name == "spectre_sources":
        g = GOLD["spectre_sources"]
        assert np.allclose(w[:, flat.index("node_1")], g["node_1"])
        assert np.allclose(w[:, flat.index("node_3")], g["node_3"])
        assert w[-1, flat.index("node_2")] == pytest.approx(g["node_2_end"])
        assert w[-1, flat.index("node_4")] == pytest.approx(g["node_4_end"])
    elif name == "pwl_current":
        ref = np.clip((t - 1e-3) / 8e-3, 0, 1) * 2 * 2
        assert np.allclose(w[:, flat.index("vout")], ref, atol=1e-7, rtol=1e-7)
    elif name == "butterworth":
        assert np.max(np.abs(w[:, flat.index("vout")] - K.butterworth_exact(t))) < GOLD["butterworth"]["tol"]


@pytest.mark.parametrize("kernel", [L.BATCH_KERNEL_AUTO, L.BATCH_KERNEL_GLOBAL])
@pytest.mark.parametrize("case", TRAN_CASES, ids=[c[0] for c in TRAN_CASES])
def test_tran_plain_reference_circuits(engine, case, kernel):
    """tran! in one launch (AUTO) and on the plain path (GLOBAL: host step
    control, one hipGraph per Newton iteration): identical steps to the oracle
    and the reference's answers."""
    name, flat, o, u0 = _tran_case(case)
    o.batch_kernel = kernel
    _say(f"plain tran {name}, kernel {kernel}")
    sol = engine.load(flat).tran(o, None, u0)
    w_ref, _, st_ref, rc = O.tran(flat, flat.params(), u0, o)
    assert sol.retcode == "Success" and rc == 0
    assert sol.stats.steps == st_ref.steps
    assert _close(sol.wave, w_ref, 1e-6, 1e-9)
    _check_reference(name, flat, o, sol.wave)


@pytest.mark.parametrize("kernel", [L.BATCH_KERNEL_LDS, L.BATCH_KERNEL_GLOBAL])
def test_batch_reference_circuits(engine, kernel):
    """The transient cases above, one batch per output grid (different
    circuits in one launch), on both batched kernels."""
    for case in TRAN_CASES:
        name, flat, o, u0 = _tran_case(case)
        _say(f"batched kernel {kernel}: {name}")
        o.batch_kernel = kernel
        p = flat.params()
        r = ch.tran_batch([flat, flat], [p, p], o, u0=None if u0 is None else [u0, u0], engine=engine)
        w_ref, _, st_ref, rc = O.tran(flat, p, u0, o)
        assert rc == 0
        for i in range(2):
            assert r.stats[i].retcode == 0, (name, i)
            assert r.stats[i].steps == st_ref.steps, name
            assert _close(r.wave[i], w_ref, 1e-6, 1e-9), name
        _check_reference(name, flat, o, r.wave[0])


def test_batch_uneven_mixed_circuits(engine):
    """Five different circuits (inductors, controlled and PWL sources,
    m-factors, MOSFETs) with UIC starts in one launch of the LDS kernel."""
    _say("batched mixed circuits")
    from cedarhip.workloads import inverter
    fns = [K.vrc, K.multi_vrc, K.butterworth, K.spice_controlled, inverter()]
    flats = [ch.lower(f) for f in fns]
    o = ch.grid_options((0.0, 2e-9), n_out=41, reltol=1e-6, abstol=1e-9, init=L.INIT_DCOP,
                        batch_kernel=L.BATCH_KERNEL_LDS)
    ps = [f.params() for f in flats]
    r = ch.tran_batch(flats, ps, o, engine=engine)
    for i, f in enumerate(flats):
        w_ref, _, st_ref, rc = O.tran(f, ps[i], None, o)
        assert rc == 0 and r.stats[i].retcode == 0, i
        assert r.stats[i].steps == st_ref.steps, i
        assert _close(r.wave[i], w_ref, 1e-6, 1e-9), i
