"""GPU parity: the HIP path (through the C-ABI) against the CPU oracle.

Bars: device stamps and assembled Jacobian /
residual within 1e-12 relative; node waveforms within reltol 1e-6 and abstol
1e-9 V at matched output times; LU solves within 1e-12 relative residual.
"""
import numpy as np
import pytest

import cedarhip as ch
from cedarhip import lib as L
from cedarhip.workloads import inverter, rc_mesh, ring_initial_state, ring_mc, ring_oscillator
from oracle import oracle as O

pytestmark = pytest.mark.gpu

RTOL_STAMP = 1e-12


def _say(msg):
    print(f"[gpu] {msg}", flush=True)


def _rel_close(a, b, rtol, atol=0.0):
    a, b = np.asarray(a), np.asarray(b)
    return np.all(np.abs(a - b) <= rtol * np.maximum(np.abs(a), np.abs(b)) + atol)


def _states(flat, rng, k=5):
    """Random operating points: node voltages in [-0.2, 2.0] V, branch currents ~1 mA."""
    out = []
    for _ in range(k):
        u = rng.uniform(-0.2, 2.0, flat.n)
        u[flat.n_nodes:] = 1e-3 * rng.standard_normal(flat.n - flat.n_nodes)
        out.append(u)
    return out


@pytest.mark.parametrize("name,circuit", [("inverter", inverter()),
                                          ("ring11", ring_oscillator(11)),
                                          ("ring51", ring_oscillator(51))])
def test_residual_jacobian_parity(engine, name, circuit):
    _say(f"residual/jacobian parity {name}")
    flat = ch.lower(circuit)
    sys = engine.load(flat)
    p = flat.params()
    rng = np.random.default_rng(7)
    proto = sys.jac_prototype
    for u in _states(flat, rng):
        du = 1e6 * rng.standard_normal(flat.n)
        for t, mode in ((0.35e-9, L.MODE_TRAN), (0.0, L.MODE_DCOP)):
            r_gpu = sys.f(None, du, u, p, t, mode)
            r_ref = O.residual(flat, p, u, du, t, mode)
            scale = np.max(np.abs(r_ref)) + 1e-30
            assert np.max(np.abs(r_gpu - r_ref)) <= RTOL_STAMP * scale, (name, mode)
            gamma = 3.7e12
            J_gpu = sys.jac_matrix(du, u, p, gamma, t, mode).toarray()
            J_ref = O.jacobian(flat, p, u, gamma, t, mode)
            scale = np.max(np.abs(J_ref))
            assert np.max(np.abs(J_gpu - J_ref)) <= RTOL_STAMP * scale, (name, mode)
            # the pattern covers every nonzero of the reference Jacobian
            assert np.all((J_ref != 0) <= (proto.toarray() != 0))


def test_lu_solve_parity(engine):
    _say("lu refactor/solve ring51")
    flat = ch.lower(ring_oscillator(51))
    sys = engine.load(flat)
    p = flat.params()
    rng = np.random.default_rng(3)
    u = _states(flat, rng, 1)[0]
    vals = sys.jac(None, None, u, p, 1e13, 0.0)
    J = sys.jac_matrix(None, u, p, 1e13, 0.0).toarray()
    sys.lu_refactor(vals)
    b = rng.standard_normal(flat.n)
    x = sys.lu_solve(b)
    assert np.linalg.norm(J @ x - b) <= 1e-12 * np.linalg.norm(J) * np.linalg.norm(x)
    xt = sys.lu_solve(b, transpose=True)
    assert np.linalg.norm(J.T @ xt - b) <= 1e-12 * np.linalg.norm(J) * np.linalg.norm(xt)
    assert _rel_close(x, np.linalg.solve(J, b), 1e-9, 1e-15)


def test_dcop_inverter(engine):
    _say("dcop inverter")
    flat = ch.lower(inverter())
    sys = engine.load(flat)
    sol = sys.dcop()
    u_ref, st, rc = O.dcop(flat, flat.params())
    assert sol.retcode == "Success" and rc == 0
    assert _rel_close(sol.u, u_ref, 1e-9, 1e-12)


@pytest.mark.parametrize("kernel", [L.BATCH_KERNEL_AUTO, L.BATCH_KERNEL_GLOBAL])
def test_tran_plain_inverter(engine, kernel):
    """Config 0 over its whole span: the inverter, 0-20 ns, BDF2 at reltol 1e-6,
    in one launch (AUTO) and on the plain path (GLOBAL)."""
    _say(f"plain tran inverter 0-20ns, kernel {kernel}")
    flat = ch.lower(inverter())
    opts = ch.grid_options((0.0, 20e-9), dt_out=10e-12, batch_kernel=kernel)
    sys = engine.load(flat)
    sol = sys.tran(opts)
    w_ref, uf_ref, st_ref, rc = O.tran(flat, flat.params(), None, opts)
    assert sol.retcode == "Success" and rc == 0
    assert sol.stats.steps == st_ref.steps
    assert _rel_close(sol.wave, w_ref, 1e-6, 1e-9)


def test_tran_batch_of_one(engine):
    """cs_tran with batch_kernel = LDS runs the circuit as a batch of one in the
    LDS-resident kernel: the inverter over the plain test's 0-20 ns span (DC
    start) and a 21-stage ring from its UIC state, against the oracle at the
    same bars; modified Newton and a supernodal circuit are refused."""
    _say("batch-of-one tran: inverter 0-20ns, 21-stage ring 0-0.5ns")
    flat = ch.lower(inverter())
    opts = ch.grid_options((0.0, 20e-9), dt_out=10e-12, batch_kernel=L.BATCH_KERNEL_LDS)
    sol = engine.load(flat).tran(opts)
    w_ref, uf_ref, st_ref, rc = O.tran(flat, flat.params(), None, opts)
    assert sol.retcode == "Success" and rc == 0
    assert sol.stats.steps == st_ref.steps
    assert _rel_close(sol.wave, w_ref, 1e-6, 1e-9)
    flats, params, u0s, stages = ring_mc(n_inst=1, seed=5, nmin=21, nmax=21)
    opts = ch.grid_options((0.0, 0.5e-9), dt_out=10e-12, init=L.INIT_UIC, batch_kernel=L.BATCH_KERNEL_LDS)
    sol = engine.load(flats[0]).tran(opts, params[0], u0s[0])
    w_ref, uf_ref, st_ref, rc = O.tran(flats[0], params[0], u0s[0], opts)
    assert sol.retcode == "Success" and rc == 0
    assert sol.stats.steps == st_ref.steps
    assert _rel_close(sol.wave, w_ref, 1e-6, 1e-9)
    np.testing.assert_allclose(sol.u_final, uf_ref, rtol=1e-6, atol=1e-9)
    with pytest.raises(ch.CedarHIPError):
        engine.load(flat).tran(ch.grid_options((0.0, 1e-10), n_out=3, jac_reuse=1,
                                               batch_kernel=L.BATCH_KERNEL_LDS))
    mesh = ch.lower(rc_mesh(8, 8, 4, seed=1))
    with pytest.raises(ch.CedarHIPError):
        engine.load(mesh, solver=L.SOLVER_SUPERNODAL).tran(
            ch.grid_options((0.0, 1e-10), n_out=3, batch_kernel=L.BATCH_KERNEL_LDS))


def test_batch_rings_parity_and_determinism(engine):
    _say("batched rings 0-0.5ns")
    flats, params, u0s, stages = ring_mc(n_inst=12, seed=5, nmin=11, nmax=31)
    opts = ch.grid_options((0.0, 0.5e-9), dt_out=10e-12, init=L.INIT_UIC)
    r1 = ch.tran_batch(flats, params, opts, u0=u0s, engine=engine)
    r2 = ch.tran_batch(flats, params, opts, u0=u0s, engine=engine)
    w_ref, uf_ref, st_ref, rc = O.tran_batch(flats, params, u0s, opts)
    assert rc == 0
    for i in range(len(flats)):
        assert r1.stats[i].retcode == 0
        assert r1.stats[i].steps == st_ref[i].steps, i
        assert _rel_close(r1.wave[i], w_ref[i], 1e-6, 1e-9), i
        assert np.array_equal(r1.wave[i], r2.wave[i]), "batched run is not bit-reproducible"


@pytest.mark.parametrize("kernel", [L.BATCH_KERNEL_LDS, L.BATCH_KERNEL_GLOBAL])
def test_batch_kernels_uneven_rings(engine, kernel):
    """Both batched kernels on uneven rings (11..101 stages: several LDS size
    classes, one and two rows per lane) against the oracle."""
    _say(f"batched kernel {kernel}: rings 11..101, 0-0.2ns")
    flats, params, u0s, stages = ring_mc(n_inst=24, seed=9, nmin=11, nmax=101)
    opts = ch.grid_options((0.0, 0.2e-9), dt_out=10e-12, init=L.INIT_UIC, batch_kernel=kernel)
    r = ch.tran_batch(flats, params, opts, u0=u0s, engine=engine)
    w_ref, uf_ref, st_ref, rc = O.tran_batch(flats, params, u0s, opts)
    assert rc == 0
    for i in range(len(flats)):
        assert r.stats[i].retcode == 0, i
        assert r.stats[i].steps == st_ref[i].steps, (i, int(stages[i]))
        assert _rel_close(r.wave[i], w_ref[i], 1e-6, 1e-9), i
        np.testing.assert_allclose(r.u_final[i], uf_ref[i], rtol=1e-6, atol=1e-9)


def test_batch_lds_inverter_dcop_pulse(engine):
    """LDS-resident kernel with DC-operating-point initialisation, a PULSE
    source and its breakpoints, against the oracle over two periods."""
    _say("LDS kernel: inverter DC op + pulse, 0-4ns")
    f = ch.lower(inverter())
    p = f.params()
    opts = ch.grid_options((0.0, 4e-9), dt_out=50e-12, init=L.INIT_DCOP,
                           batch_kernel=L.BATCH_KERNEL_LDS)
    r = ch.tran_batch([f, f], [p, p], opts, engine=engine)
    w_ref, uf_ref, st_ref, rc = O.tran_batch([f], [p], None, opts)
    assert rc == 0
    for i in range(2):
        assert r.stats[i].retcode == 0
        assert r.stats[i].steps == st_ref[0].steps
        assert _rel_close(r.wave[i], w_ref[0], 1e-6, 1e-9)
    assert np.array_equal(r.wave[0], r.wave[1])


def test_batch_rings_full_span(engine):
    """Config 2's span on rings of 11 to 101 stages (both ends included):
    0-10 ns on the packed LDS kernel (150 k to 200 k steps per instance),
    waveforms every 10 ps against the oracle's by the long-span bar of
    spans.py: step counts within 1e-4, every sample within reltol/abstol plus
    a 2e-16 s edge shift, half-supply crossing times within 2e-16 s."""
    from spans import assert_same_waveform
    _say("batched rings 11..101, 0-10ns")
    flats, params, u0s, stages = ring_mc(n_inst=10, seed=21, nmin=11, nmax=101)
    extra = [11, 101]
    for nst in extra:
        flat = ch.lower(ring_oscillator(nst))
        rng = np.random.default_rng(nst)
        p = flat.params()
        lay = flat.layout()
        p[lay["mos_vth"]:lay["mos_vth"] + 2 * nst] += 0.03 * rng.standard_normal(2 * nst)
        flats.append(flat)
        params.append(p)
        u0s.append(ring_initial_state(flat, rng))
        stages = np.append(stages, nst)
    opts = ch.grid_options((0.0, 10e-9), dt_out=10e-12, init=L.INIT_UIC, batch_kernel=L.BATCH_KERNEL_LDS)
    r = ch.tran_batch(flats, params, opts, u0=u0s, engine=engine)
    w_ref, uf_ref, st_ref, rc = O.tran_batch(flats, params, u0s, opts)
    assert rc == 0
    assert 11 in set(int(x) for x in stages) and 101 in set(int(x) for x in stages)
    t = opts.t_start + np.arange(opts.n_out) * opts.dt_out
    for i in range(len(flats)):
        assert r.stats[i].retcode == 0, i
        assert_same_waveform(r.wave[i], w_ref[i], t, r.stats[i].steps, st_ref[i].steps, 0.9,
                             flats[i].n_nodes, what=(i, int(stages[i])))


def test_batch_inverter_full_span(engine):
    """Config 0 on both batched kernels: 0-20 ns from the DC operating point."""
    _say("batched inverter 0-20ns")
    f = ch.lower(inverter())
    p = f.params()
    w_ref, _, st_ref, rc = None, None, None, None
    for kernel in (L.BATCH_KERNEL_LDS, L.BATCH_KERNEL_GLOBAL):
        opts = ch.grid_options((0.0, 20e-9), dt_out=10e-12, init=L.INIT_DCOP, batch_kernel=kernel)
        if w_ref is None:
            w_ref, _, st_ref, rc = O.tran_batch([f], [p], None, opts)
            assert rc == 0
        r = ch.tran_batch([f], [p], opts, engine=engine)
        assert r.stats[0].retcode == 0
        assert r.stats[0].steps == st_ref[0].steps
        assert _rel_close(r.wave[0], w_ref[0], 1e-6, 1e-9)
