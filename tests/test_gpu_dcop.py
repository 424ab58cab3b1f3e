"""GPU DC operating point: CedarDCOp's trajectories (src/dcop.jl:53-94) and
the gmin ladder on every path - the one launch and the plain path (cs_dcop,
cs_tran), supernodal, and both batched kernels (INIT_DCOP) - against the
oracle and the closed form."""
import numpy as np
import pytest

import cedarhip as ch
from cedarhip import lib as L
from oracle import oracle as O

import circuits as K

pytestmark = pytest.mark.gpu

CASES = [("restart_vth0", 0.0), ("gmin_ladder_vth04", 0.4)]


KERNELS = [L.BATCH_KERNEL_AUTO, L.BATCH_KERNEL_GLOBAL]   # the one launch (where a circuit fits), the plain path


@pytest.mark.parametrize("name,vth", CASES)
@pytest.mark.parametrize("solver", [L.SOLVER_LEVEL, L.SOLVER_SUPERNODAL])
@pytest.mark.parametrize("kernel", KERNELS)
def test_dcop_restarts_plain(engine, name, vth, solver, kernel):
    print(f"[gpu] dcop {name} solver {solver} kernel {kernel}", flush=True)
    flat = ch.lower(K.diode_nmos(vth), gmin=0.0)
    sol = engine.load(flat, solver=solver).dcop(opts=ch.TranOptions(batch_kernel=kernel))
    u_ref, _, rc = O.dcop(flat, flat.params())
    assert rc == 0 and sol.retcode == "Success"
    assert sol["a"] == pytest.approx(K.diode_nmos_exact(vth), abs=1e-6)
    assert sol["a"] == pytest.approx(u_ref[flat.index("a")], abs=1e-9)


@pytest.mark.parametrize("kernel", [L.BATCH_KERNEL_LDS, L.BATCH_KERNEL_GLOBAL])
def test_dcop_restarts_batched(engine, kernel):
    """Both circuits and the failing one in one batch: per-instance DC
    operating points, then a short transient; the failing instance reports
    InitialFailure and does not stop the others."""
    print(f"[gpu] batched dcop kernel {kernel}", flush=True)
    flats = [ch.lower(K.diode_nmos(v), gmin=0.0) for _, v in CASES] + [ch.lower(K.floating_cap)]
    ps = [f.params() for f in flats]
    o = ch.grid_options((0.0, 1e-9), n_out=11, init=L.INIT_DCOP, batch_kernel=kernel)
    r = ch.tran_batch(flats, ps, o, engine=engine)
    for i, (_, vth) in enumerate(CASES):
        w_ref, _, st_ref, rc = O.tran(flats[i], ps[i], None, o)
        assert rc == 0 and r.stats[i].retcode == 0, i
        assert r.wave[i][0, 0] == pytest.approx(K.diode_nmos_exact(vth), abs=1e-6)
        assert np.allclose(r.wave[i], w_ref, rtol=1e-6, atol=1e-9)
    assert r.retcodes[2] == "InitialFailure"


@pytest.mark.parametrize("kernel", KERNELS)
def test_dcop_failure_plain(engine, kernel):
    print(f"[gpu] dcop failure plain, kernel {kernel}", flush=True)
    flat = ch.lower(K.floating_cap)
    sys = engine.load(flat)
    assert sys.dcop(opts=ch.TranOptions(batch_kernel=kernel)).retcode == "InitialFailure"
    sol = sys.tran(ch.grid_options((0.0, 1e-9), n_out=11, batch_kernel=kernel))
    assert sol.retcode == "InitialFailure"
