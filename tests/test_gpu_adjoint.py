"""GPU adjoint (cs_adjoint_batch) against the oracle and finite differences.

The GPU records its accepted-step sequence; the oracle replays exactly that
sequence (same discrete scheme) for (a) its own adjoint and (b) central finite
differences in each width (h = 1e-6 relative).  Bars: energy to 1e-9
relative, gradients to 1e-6 against the oracle adjoint and 1e-5 against the
finite differences.  Runs are bounded (max_steps counts accepted plus
rejected steps) so that a failing case ends with an error code.
"""
import numpy as np
import pytest

import cedarhip as ch
from cedarhip.workloads import ring_initial_state, ring_oscillator
from oracle import oracle as O

pytestmark = pytest.mark.gpu

T_STOP = 0.3e-9


def _say(msg):
    print(f"[gpu] {msg}", flush=True)


def _batch(sizes, seed):
    rng = np.random.default_rng(seed)
    cache, flats, params, u0s = {}, [], [], []
    for N in sizes:
        if N not in cache:
            cache[N] = ch.lower(ring_oscillator(N))
        f = cache[N]
        p = f.params()
        lay = f.layout()
        nm = len(f.arrays["mos_w"])
        p[lay["mos_w"]:lay["mos_w"] + nm] = rng.uniform(0.5e-6, 4e-6, nm)
        flats.append(f)
        params.append(p)
        u0s.append(ring_initial_state(f, rng))
    return flats, params, u0s


NTOL = 1e-8


def _opts():
    return ch.TranOptions(t_start=0.0, t_stop=T_STOP, reltol=1e-6, abstol=1e-9,
                          newton_tol=NTOL, newton_maxit=30, init=1, max_steps=60_000)


def test_adjoint_matches_oracle_and_fd(engine):
    _say("adjoint rings 5/7/11, 0.3 ns")
    flats, params, u0s = _batch([5, 7, 11, 5], seed=4)
    o = _opts()
    res = ch.adjoint_batch(flats, params, u0s, o, vsrc=0, ckpt_every=64, keep_logs=True,
                           max_steps=40_000, engine=engine)
    _say(f"adjoint done: {res.retcodes}, steps {list(res.n_steps)}, {res.kernel_ms:.1f} ms")
    assert all(r == "Success" for r in res.retcodes), res.retcodes
    oo = dict(t_start=0.0, t_stop=T_STOP, reltol=1e-6, abstol=1e-9, newton_tol=NTOL,
              newton_maxit=30, init=1)
    for i, f in enumerate(flats):
        tl, npl = res.t_logs[i], res.npts_logs[i]
        E_or, g_or, rc = O.adjoint_replay(f, params[i], u0s[i], tl, npl, 0, **oo)
        assert rc == 0
        assert res.energy[i] == pytest.approx(E_or, rel=1e-9)
        np.testing.assert_allclose(res.grads[i], g_or, rtol=1e-6, atol=1e-6 * np.max(np.abs(g_or)))
        lay = f.layout()
        for k in (0, 1, len(g_or) - 1):
            p = params[i]
            hW = 1e-6 * p[lay["mos_w"] + k]
            pp, pm = p.copy(), p.copy()
            pp[lay["mos_w"] + k] += hW
            pm[lay["mos_w"] + k] -= hW
            Ep, _ = O.replay_energy(f, pp, u0s[i], tl, npl, 0, **oo)
            Em, _ = O.replay_energy(f, pm, u0s[i], tl, npl, 0, **oo)
            fd = (Ep - Em) / (2 * hW)
            assert res.grads[i][k] == pytest.approx(fd, rel=1e-5), (i, k)


def test_adjoint_checkpoint_interval_and_determinism(engine):
    _say("adjoint checkpoint interval 64 vs 7, repeat")
    flats, params, u0s = _batch([7, 9], seed=8)
    o = _opts()
    r64 = ch.adjoint_batch(flats, params, u0s, o, ckpt_every=64, max_steps=40_000, engine=engine)
    r7 = ch.adjoint_batch(flats, params, u0s, o, ckpt_every=7, max_steps=40_000, engine=engine)
    r64b = ch.adjoint_batch(flats, params, u0s, o, ckpt_every=64, max_steps=40_000, engine=engine)
    _say(f"adjoint runs done: {r64.kernel_ms:.1f} / {r7.kernel_ms:.1f} / {r64b.kernel_ms:.1f} ms")
    for i in range(len(flats)):
        assert np.array_equal(r64.grads[i], r64b.grads[i]), "adjoint is not bit-reproducible"
        assert r64.energy[i] == r64b.energy[i]
        # recomputation from a checkpoint replays the same Newton iterates, so
        # the checkpoint interval does not change a bit
        assert np.array_equal(r7.grads[i], r64.grads[i])
        assert r7.energy[i] == r64.energy[i]


def test_adjoint_config_51_stage_full_span(engine):
    """The adjoint workload itself: 51-stage rings with all 102 widths drawn
    from U[0.5, 4] um, supply energy over the full 0-5 ns, checkpoints every 64
    accepted steps.  All 102 gradients of each instance against the oracle's
    adjoint on the GPU's step sequence (1e-6), three widths per instance
    against central differences h = 1e-6 W on that sequence (1e-5)."""
    from concurrent.futures import ThreadPoolExecutor

    from cedarhip.workloads import ring_widths
    _say("adjoint 4 x 51-stage rings, 0-5 ns")
    flats, params, u0s = ring_widths(n_inst=4, nstage=51, seed=7)
    o = ch.TranOptions(t_start=0.0, t_stop=5e-9, reltol=1e-6, abstol=1e-9, newton_tol=1e-6,
                       newton_maxit=30, init=1, max_steps=400_000)
    res = ch.adjoint_batch(flats, params, u0s, o, vsrc=0, ckpt_every=64, keep_logs=True,
                           max_steps=300_000, engine=engine)
    _say(f"adjoint done: {res.retcodes}, steps {list(res.n_steps)}, {res.kernel_ms:.1f} ms")
    assert all(r == "Success" for r in res.retcodes), res.retcodes
    oo = dict(t_start=0.0, t_stop=5e-9, reltol=1e-6, abstol=1e-9, newton_tol=1e-6, newton_maxit=30,
              init=1)
    lay = flats[0].layout()
    jobs = []
    for i, f in enumerate(flats):
        tl, npl = res.t_logs[i], res.npts_logs[i]
        jobs.append(("adj", i, None))
        for k in (0, 51, 101):
            jobs.append(("fd", i, k))

    def run(job):
        kind, i, k = job
        f, p, tl, npl = flats[i], params[i], res.t_logs[i], res.npts_logs[i]
        if kind == "adj":
            return O.adjoint_replay(f, p, u0s[i], tl, npl, 0, **oo)
        hW = 1e-6 * p[lay["mos_w"] + k]
        pp, pm = p.copy(), p.copy()
        pp[lay["mos_w"] + k] += hW
        pm[lay["mos_w"] + k] -= hW
        Ep, _ = O.replay_energy(f, pp, u0s[i], tl, npl, 0, **oo)
        Em, _ = O.replay_energy(f, pm, u0s[i], tl, npl, 0, **oo)
        return (Ep - Em) / (2 * hW)

    with ThreadPoolExecutor(max_workers=12) as ex:
        out = list(ex.map(run, jobs))
    for job, r in zip(jobs, out):
        kind, i, k = job
        if kind == "adj":
            E_or, g_or, rc = r
            assert rc == 0
            assert len(g_or) == 102
            assert res.energy[i] == pytest.approx(E_or, rel=1e-9)
            np.testing.assert_allclose(res.grads[i], g_or, rtol=1e-6, atol=1e-6 * np.max(np.abs(g_or)))
        else:
            assert res.grads[i][k] == pytest.approx(r, rel=1e-5), (i, k)


@pytest.mark.parametrize("n", [201, 215, 217, 225, 251])
def test_adjoint_around_64k_of_lds(engine, n):
    """Rings whose reverse kernel needs 61 to 76 KB of LDS, on both sides of
    64 KiB (between 215 and 217 stages), two of them beside a small one:
    energy and gradients against the oracle's adjoint on the GPU's steps."""
    _say(f"adjoint {n}-stage ring, 2 ps")
    flats, params, u0s = _batch([n, 5, n], seed=n)
    kw = dict(t_start=0.0, t_stop=2e-12, reltol=1e-6, abstol=1e-9, newton_tol=NTOL, newton_maxit=30, init=1)
    res = ch.adjoint_batch(flats, params, u0s, ch.TranOptions(max_steps=2000, **kw), vsrc=0, ckpt_every=16,
                           keep_logs=True, max_steps=1000, engine=engine)
    assert all(r == "Success" for r in res.retcodes), res.retcodes
    for i, f in enumerate(flats):
        E_or, g_or, rc = O.adjoint_replay(f, params[i], u0s[i], res.t_logs[i], res.npts_logs[i], 0, **kw)
        assert rc == 0
        assert res.energy[i] == pytest.approx(E_or, rel=1e-9)
        np.testing.assert_allclose(res.grads[i], g_or, rtol=1e-6, atol=1e-6 * np.max(np.abs(g_or)))


def test_adjoint_forward_residency(engine):
    """185-stage rings: three instances of the forward kernel fit a CU's LDS and
    two of the reverse kernel, so 768 of them take one round forward and two
    back; with both kernels at the reverse's size they took twice the time of
    512 (one round each way)."""
    _say("adjoint residency, 185-stage rings")
    flat = ch.lower(ring_oscillator(185))
    p, u0 = flat.params(), ring_initial_state(flat, np.random.default_rng(2))
    o = ch.TranOptions(t_stop=2e-12, init=1)
    ms = {}
    for count in (512, 768):
        for _ in range(2):
            r = ch.adjoint_batch([flat] * count, [p] * count, [u0] * count, o, max_steps=1000, engine=engine)
        assert set(r.retcodes) == {"Success"}
        ms[count] = r.kernel_ms
    _say(f"kernel ms {ms}")
    assert ms[768] <= 1.75 * ms[512]
