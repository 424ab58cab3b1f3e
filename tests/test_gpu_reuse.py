"""Modified Newton (cs_tran_opts.jac_reuse = 1: the step's first factors
reused by its later Newton iterations, IDA's Jacobian reuse, src/sweeps.jl:456)
on cs_tran, level-scheduled and supernodal, against the oracle running the
same rule (or_tran with jac_reuse).

Modified Newton's iterates depend on how many iterations a step took, and an
update at the convergence threshold can take one more iteration on one side
(the two LUs round differently); from there the step sequences part, as they
do over long spans with full Newton.  The bar for the nonlinear circuits is
therefore the long-span one (spans.py): step counts within 1e-4, samples
within sqrt(n) (reltol |u| + abstol) plus a 2e-16 s edge shift, half-supply
crossings within 2e-16 s.  A linear circuit has a constant Jacobian, so there
modified and full Newton take the same iterates: the Butterworth waveform is
identical bit for bit.  The batched kernels and the adjoint refuse the
option.
"""
import numpy as np
import pytest

import cedarhip as ch
from cedarhip import lib as L
from cedarhip.workloads import inverter, rc_mesh, ring_mc
from oracle import oracle as O

import circuits as K
from spans import assert_same_waveform

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[gpu] {msg}", flush=True)


def test_reuse_rings_plain(engine):
    _say("jac_reuse: plain path, rings, 0-0.5ns")
    flats, params, u0s, stages = ring_mc(n_inst=3, seed=31, nmin=11, nmax=101)
    for f, p, u0, nst in zip(flats, params, u0s, stages):
        s = engine.load(f, solver=L.SOLVER_LEVEL)
        o = ch.grid_options((0.0, 0.5e-9), dt_out=10e-12, init=L.INIT_UIC, jac_reuse=1)
        sol = s.tran(o, p, u0)
        w, _, st, rc = O.tran(f, p, u0, o, probes=s.probes)
        assert sol.retcode == "Success" and rc == 0
        assert abs(sol.stats.newton_iters - st.newton_iters) <= 1e-3 * st.newton_iters
        t = o.t_start + np.arange(o.n_out) * o.dt_out
        assert_same_waveform(sol.wave, w, t, sol.stats.steps, st.steps, 0.9, f.n_nodes, what=int(nst))


def test_reuse_inverter_and_filter_plain(engine):
    _say("jac_reuse: plain path, inverter DC op + pulse 0-4ns, Butterworth 0-4s")
    f = ch.lower(inverter())
    p = f.params()
    s = engine.load(f, solver=L.SOLVER_LEVEL)
    o = ch.grid_options((0.0, 4e-9), dt_out=50e-12, jac_reuse=1)
    sol = s.tran(o, p)
    w, _, st, rc = O.tran(f, p, None, o, probes=s.probes)
    assert sol.retcode == "Success" and rc == 0
    t = o.t_start + np.arange(o.n_out) * o.dt_out
    assert_same_waveform(sol.wave, w, t, sol.stats.steps, st.steps, 0.9, f.n_nodes)

    fb = ch.lower(K.butterworth)
    sb = engine.load(fb, solver=L.SOLVER_LEVEL)
    u0 = np.zeros(fb.n)
    for kernel in (L.BATCH_KERNEL_AUTO, L.BATCH_KERNEL_GLOBAL):   # the one launch, the plain path
        ob = ch.grid_options((0.0, 4.0), n_out=41, init=L.INIT_UIC, batch_kernel=kernel)
        full = sb.tran(ob, u0=u0)
        ob.jac_reuse = 1
        mod = sb.tran(ob, u0=u0)
        assert mod.retcode == "Success" and mod.stats.steps == full.stats.steps
        assert mod.stats.newton_iters == full.stats.newton_iters
        assert np.array_equal(np.asarray(mod.wave), np.asarray(full.wave))


def test_reuse_power_grid_supernodal(engine):
    _say("jac_reuse: supernodal path, 12x12 grid 0-5ns")
    f = rc_mesh(12, 12, 12, seed=2)
    s = engine.load(f, solver=L.SOLVER_SUPERNODAL)
    p = f.params()
    o = ch.TranOptions(t_start=0.0, t_stop=5e-9, reltol=1e-6, abstol=1e-9, n_out=501, dt_out=1e-11, jac_reuse=1)
    sol = s.tran(o, p)
    w, _, st, rc = O.tran(f, p, None, o, probes=s.probes)
    _say(f"  {sol.stats.steps} steps (oracle {st.steps}), {sol.stats.newton_iters} iterations "
         f"(oracle {st.newton_iters})")
    assert sol.retcode == "Success" and rc == 0
    t = o.t_start + np.arange(o.n_out) * o.dt_out
    assert_same_waveform(sol.wave, w, t, sol.stats.steps, st.steps, 0.5, f.n_nodes)
    full = s.tran(ch.TranOptions(t_start=0.0, t_stop=5e-9, reltol=1e-6, abstol=1e-9, n_out=501, dt_out=1e-11), p)
    assert full.retcode == "Success"
    assert abs(sol.stats.newton_iters - full.stats.newton_iters) <= 0.05 * full.stats.newton_iters


def test_reuse_refused_in_batches(engine):
    f = ch.lower(inverter())
    p = f.params()
    for kern in (L.BATCH_KERNEL_LDS, L.BATCH_KERNEL_GLOBAL):
        og = ch.grid_options((0.0, 1e-10), n_out=3, jac_reuse=1, batch_kernel=kern)
        with pytest.raises(ch.CedarHIPError):
            ch.tran_batch([f], [p], og, engine=engine)
    s = engine.load(f)
    with pytest.raises(ch.CedarHIPError):
        s.tran(ch.grid_options((0.0, 1e-10), n_out=3, jac_reuse=2), p)
