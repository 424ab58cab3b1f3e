"""SPICE decks on the GPU: the reference's own decks (tests/golden/
spice_decks.json, from test/basic.jl) through cs_dcop / cs_tran and the
batched kernels, and a ring-oscillator deck through the LDS-resident batched
kernel, against the oracle and the reference's answers."""
import json
import os

import numpy as np
import pytest

import cedarhip as ch
from cedarhip import lib as L
from cedarhip.spice import make_spice_circuit
from cedarhip.workloads import ring_initial_state, ring_spice
from oracle import oracle as O

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))
DECKS = json.load(open(os.path.join(HERE, "golden", "spice_decks.json")))
MODELS_DIR = os.path.join(os.path.dirname(HERE), "cedarsim.jl_amd", "models")


@pytest.mark.parametrize("name", ["spice_sources", "subcircuits", "multiplicities"])
def test_spice_dc_on_device(engine, name):
    print(f"[gpu] spice dc {name}", flush=True)
    flat = ch.lower(make_spice_circuit(DECKS[name]["deck"]))
    sol = engine.load(flat).dcop()
    assert sol.retcode == "Success"
    for k, v in DECKS[name]["dc"].items():
        assert sol[k] == pytest.approx(v, rel=1e-12, abs=1e-12), k


@pytest.mark.parametrize("name", ["dynamic_scope", "default_temper"])
def test_spice_scopes_on_device(engine, name):
    print(f"[gpu] spice scope {name}", flush=True)
    flat = ch.lower(make_spice_circuit(DECKS[name]["deck"]))
    sol = engine.load(flat).dcop()
    for dev, v_exp in DECKS[name]["voltage"].items():
        kind, k = flat.device_names[dev]
        a, b = flat.arrays["res_nodes"][2 * k:2 * k + 2]
        v = (sol.u[a] if a >= 0 else 0.0) - (sol.u[b] if b >= 0 else 0.0)
        assert v == pytest.approx(v_exp, rel=1e-9)


def test_multimode_source_on_device(engine):
    """test/basic.jl:534-553: DC 5 with SIN(10 3 1k); the transient starts on
    the waveform (CedarDCOp's DC point, then the consistent start at t0) on
    the one launch, the plain path and both batched kernels."""
    print("[gpu] spice multimode source", flush=True)
    flat = ch.lower(make_spice_circuit(DECKS["multimode_source"]["deck"]))
    o = ch.grid_options((0.0, 1e-3), n_out=21, reltol=1e-8, abstol=1e-10)
    w_ref, _, st_ref, rc = O.tran(flat, flat.params(), None, o)
    assert rc == 0 and w_ref[0, flat.index("node_vcc")] == pytest.approx(10.0)
    for kernel in (L.BATCH_KERNEL_AUTO, L.BATCH_KERNEL_GLOBAL):
        o.batch_kernel = kernel
        sol = engine.load(flat).tran(o)
        assert sol.retcode == "Success" and sol.stats.steps == st_ref.steps
        assert np.allclose(sol.wave, w_ref, rtol=1e-6, atol=1e-9)
    for kernel in (L.BATCH_KERNEL_LDS, L.BATCH_KERNEL_GLOBAL):
        o.batch_kernel = kernel
        r = ch.tran_batch([flat], [flat.params()], o, engine=engine)
        assert r.stats[0].retcode == 0 and r.stats[0].steps == st_ref.steps
        assert np.allclose(r.wave[0], w_ref, rtol=1e-6, atol=1e-9)


def test_ring_deck_on_lds_kernel(engine):
    """An 11-stage ring written as a SPICE deck (square-law devices through
    .hdl "sqlaw.va") on the LDS-resident batched kernel, 0-2 ns."""
    print("[gpu] spice ring deck", flush=True)
    fn = make_spice_circuit(ring_spice(11), None, include_dirs=[MODELS_DIR])
    flat = ch.lower(fn)
    rng = np.random.default_rng(3)
    u0 = np.zeros(flat.n)
    u0[flat.index("node_vdd")] = 1.8
    for k in range(11):
        u0[flat.index(f"node_s{k}")] = 1.8 * (k % 2) + 1e-3 * rng.standard_normal()
    o = ch.grid_options((0.0, 2e-9), dt_out=10e-12, init=L.INIT_UIC, batch_kernel=L.BATCH_KERNEL_LDS)
    r = ch.tran_batch([flat], [flat.params()], o, u0=[u0], engine=engine)
    w_ref, _, st_ref, rc = O.tran(flat, flat.params(), u0, o)
    assert rc == 0 and r.stats[0].retcode == 0
    # 40 k steps: the long-span bar (step counts within 1e-4, samples within
    # reltol/abstol plus a 2e-16 s edge shift, crossing times within 2e-16 s)
    from spans import assert_same_waveform
    t = o.t_start + np.arange(o.n_out) * o.dt_out
    assert_same_waveform(r.wave[0], w_ref, t, r.stats[0].steps, st_ref.steps, 0.9, flat.n_nodes)
