"""The packed launch's shapes against the oracle: instances per workgroup (one
for a batch below the CU count, up to eight), the two register budgets (a
batch past eight instances per CU takes the one for sixteen wavefronts), DC
and driven sources, one, two and four rows per lane, and circuits whose solve
has long tasks and updated diagonals (an RC mesh).  The step sequences are
equal, so waveforms agree to reltol 1e-6 / abstol 1e-9 V as in the other
parity tests."""
import numpy as np
import pytest

import cedarhip as ch
from cedarhip import lib as L
from cedarhip.workloads import inverter, rc_mesh, ring_initial_state, ring_oscillator
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
