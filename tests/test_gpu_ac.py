"""cs_ac / cs_noise on the GPU against the oracle (dense complex solves,
oracle.ac_response / noise_psd, themselves pinned by test/ac.jl in
test_oracle_ac.py) and against the reference's own answers: the
Butterworth of test/ac.jl (analytic H, ngspice noise table), a
common-source amplifier (device stamps in G), and RC meshes large enough
for the 256-thread kernel.  Bars: responses within 1e-12 of max |X| per
frequency, PSDs within 1e-10 relative."""
import json
import os

import numpy as np
import pytest

import cedarhip as ch
from cedarhip import lib as L
from cedarhip.spice import make_spice_circuit
from oracle import oracle as O

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
FIX = json.load(open(os.path.join(HERE, "golden", "ac_butterworth.json")))


def _say(msg):
    print(f"[gpu] {msg}", flush=True)


def _close_rows(X, R, rtol):
    scale = np.max(np.abs(R), axis=1, keepdims=True) + 1e-300
    return np.all(np.abs(X - R) <= rtol * scale)


def test_butterworth_ac_and_noise(engine):
    _say("ac/noise butterworth (test/ac.jl)")
    flat = ch.lower(make_spice_circuit(FIX["deck"]))
    sys_ = engine.load(flat, solver=L.SOLVER_LEVEL)
    dc = sys_.dcop()
    assert dc.retcode == "Success"
    tab = np.array(FIX["ngspice_hz_sqrtpsd"])
    ws = 2 * np.pi * tab[:, 0]
    obs = ["node_vout", "node_vin", "node_n1"]
    X = sys_.ac(dc.u, ws, obs)
    R = O.ac_response(flat, flat.params(), dc.u, ws, [flat.index(o) for o in obs])
    assert _close_rows(X, R, 1e-12)
    s = 1j * ws
    np.testing.assert_allclose(X[:, 0], 1.0 / ((s + 1) * (s * s + s + 1)), rtol=1e-10)
    np.testing.assert_allclose(X[:, 1], 1.0, rtol=1e-12)
    psd = sys_.noise(dc.u, ws, "node_vout", temp_c=FIX["temp_c"])
    psd_ref = O.noise_psd(flat, flat.params(), dc.u, ws, flat.index("node_vout"), temp_c=FIX["temp_c"])
    np.testing.assert_allclose(psd, psd_ref, rtol=1e-10)
    assert np.linalg.norm(np.sqrt(psd) - tab[:, 1]) <= 1e-6 * np.linalg.norm(tab[:, 1])
    # the reference's API shape: ac!(circ) then freqresp, noise!(circ) then PSD
    acs = ch.ac(flat, engine=engine)
    np.testing.assert_allclose(acs.freqresp("node_vout", ws), X[:, 0], rtol=1e-14)
    nz = ch.noise(flat, temp_c=FIX["temp_c"], engine=engine)
    np.testing.assert_allclose(nz.psd("node_vout", ws), psd, rtol=1e-14)


def test_common_source_amplifier(engine):
    """Square-law NMOS with a resistive load, biased by a DC gate source
    carrying the AC input: the small-signal gain -gm R (and its roll-off
    with a load capacitor) comes from the device's Jacobian stamps."""
    _say("ac common-source amplifier")
    deck = ("* common-source amplifier\n"
            ".hdl \"sqlaw.va\"\n"
            "VDD vdd 0 1.8\n"
            "VG g 0 DC 0.7 AC 1\n"
            "RL vdd d 5k\n"
            "CL d 0 100f\n"
            "X1 d g 0 0 sqlaw type=1 vth=0.4 kp=200u w=1u l=0.18u\n")
    fn = make_spice_circuit(deck, None, include_dirs=[os.path.join(HERE, "..", "cedarsim.jl_amd", "models")])
    flat = ch.lower(fn)
    sys_ = engine.load(flat, solver=L.SOLVER_LEVEL)
    dc = sys_.dcop()
    assert dc.retcode == "Success"
    ws = np.logspace(6, 11, 31)
    obs = ["node_d", "node_g"]
    X = sys_.ac(dc.u, ws, obs)
    R = O.ac_response(flat, flat.params(), dc.u, ws, [flat.index(o) for o in obs])
    assert _close_rows(X, R, 1e-12)
    assert abs(X[0, 0]) > 1.0   # gain at low frequency
    psd = sys_.noise(dc.u, ws, "node_d")
    psd_ref = O.noise_psd(flat, flat.params(), dc.u, ws, flat.index("node_d"))
    np.testing.assert_allclose(psd, psd_ref, rtol=1e-10)


def _mesh(nx, ny, seed):
    def ckt():
        rng = np.random.default_rng(seed)
        gnd = ch.Named(ch.net, "gnd")()
        nd = [[ch.Named(ch.net, f"n{i}_{j}")() for j in range(ny)] for i in range(nx)]
        ch.Named(ch.CurrentSource(dc=0.0, ac=1.0), "Iin")(gnd, nd[0][0])
        for i in range(nx):
            for j in range(ny):
                if i + 1 < nx:
                    ch.Named(ch.R(rng.uniform(0.5, 2.0)), f"Rx{i}_{j}")(nd[i][j], nd[i + 1][j])
                if j + 1 < ny:
                    ch.Named(ch.R(rng.uniform(0.5, 2.0)), f"Ry{i}_{j}")(nd[i][j], nd[i][j + 1])
                ch.Named(ch.C(rng.uniform(1e-12, 1e-11)), f"C{i}_{j}")(nd[i][j], gnd)
        ch.Named(ch.R(50.0), "Rt")(nd[nx - 1][ny - 1], gnd)
        ch.Gnd()(gnd)
    return ckt


@pytest.mark.parametrize("nx,ny", [(6, 7), (25, 24)])
def test_rc_mesh_ac_and_noise(engine, nx, ny):
    _say(f"ac/noise rc mesh {nx}x{ny}")
    flat = ch.lower(_mesh(nx, ny, nx * 100 + ny))
    sys_ = engine.load(flat, solver=L.SOLVER_LEVEL)
    dc = sys_.dcop()
    assert dc.retcode == "Success"
    ws = np.logspace(7, 12, 11)
    obs = [f"n0_0", f"n{nx // 2}_{ny // 2}", f"n{nx - 1}_{ny - 1}"]
    X = sys_.ac(dc.u, ws, obs)
    R = O.ac_response(flat, flat.params(), dc.u, ws, [flat.index(o) for o in obs])
    assert _close_rows(X, R, 1e-12)
    o = flat.index(obs[-1])
    psd = sys_.noise(dc.u, ws, o)
    if flat.n <= 100:
        ref = O.noise_psd(flat, flat.params(), dc.u, ws, o)
    else:
        # one transposed dense solve per frequency (the oracle's per-source
        # loop is the same sum, one solve per resistor)
        a = flat.arrays
        lay = flat.layout()
        G = O.jacobian(flat, flat.params(), dc.u, 0.0, 0.0, L.MODE_DCOP)
        Cm = O.cmatrix(flat, flat.params(), dc.u)
        kT = 1.380649e-23 * 300.15
        ref = np.zeros(len(ws))
        e = np.zeros(flat.n)
        e[o] = 1.0
        nres = len(a["res_r"])
        na = a["res_nodes"][0::2]
        nb = a["res_nodes"][1::2]
        pwr = 4 * kT / flat.params()[lay["res_r"]:lay["res_r"] + nres]
        for f, w in enumerate(ws):
            y = np.linalg.solve((G + 1j * w * Cm).T, e)
            ya = np.where(na >= 0, y[np.maximum(na, 0)], 0)
            yb = np.where(nb >= 0, y[np.maximum(nb, 0)], 0)
            ref[f] = np.sum(pwr * np.abs(ya - yb) ** 2)
    np.testing.assert_allclose(psd, ref, rtol=1e-10)


@pytest.mark.parametrize("nx,ny,nf", [(1, 1, 3), (8, 8, 7), (13, 5, 1100), (12, 12, 9), (16, 15, 9), (20, 19, 9)])
def test_ac_kernel_forms(engine, nx, ny, nf):
    """Sizes around the kernel's choices: one unknown, 64 and 65 (a level fills
    the wavefront or not), meshes that keep a frequency in LDS and that do
    not, and more frequencies than workgroups.  A dense complex solve of the
    same G + jwC bounds the difference by the condition of a passive mesh
    (below 1e2 at these values) times 6 n units of rounding: 1e-12 with room."""
    flat = ch.lower(_mesh(nx, ny, nx * 100 + ny))
    sys_ = engine.load(flat, solver=L.SOLVER_LEVEL)
    dc = sys_.dcop()
    ws = np.logspace(7, 12, nf)
    obs = ["n0_0", f"n{nx - 1}_{ny - 1}"]
    X = sys_.ac(dc.u, ws, obs)
    o = flat.index(obs[-1])
    psd = sys_.noise(dc.u, ws, o)
    G = O.jacobian(flat, flat.params(), dc.u, 0.0, 0.0, L.MODE_DCOP)
    Cm = O.cmatrix(flat, flat.params(), dc.u)
    rows = flat.arrays["res_nodes"].reshape(-1, 2)
    r = flat.params()[flat.layout()["res_r"]:][:len(rows)]
    b = np.zeros(flat.n)
    b[flat.index("n0_0")] = 1.0
    e = np.zeros(flat.n)
    e[o] = 1.0
    for k in range(0, nf, max(1, nf // 11)):
        J = G + 1j * ws[k] * Cm
        x = np.linalg.solve(J, b)
        got, ref = X[k], x[[flat.index(q) for q in obs]]
        assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(x)), (k, got, ref)
        y = np.append(np.linalg.solve(J.T, e), 0.0)   # -1: ground
        ref = np.sum(4 * 1.380649e-23 * 300.15 / r * np.abs(y[rows[:, 0]] - y[rows[:, 1]]) ** 2)
        assert abs(psd[k] - ref) <= 1e-10 * ref
