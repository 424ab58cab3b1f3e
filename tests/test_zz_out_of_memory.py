"""Calls that need no device memory for their samples on the plain path still
work when there is none for the one launch: cs_tran and cs_tran_sens fall back,
an explicit choice of the one launch reports CS_E_OOM, and nothing of the failed
allocation shows in later calls.  The memory is taken with hipMalloc from the
runtime the library links, never touched, and given back."""
import ctypes

import numpy as np
import pytest

import cedarhip as ch
from cedarhip import lib as L
from cedarhip.workloads import inverter

pytestmark = pytest.mark.gpu

MIB = 1 << 20


class _Fill:
    """All device memory but less than 40 MiB in one piece."""

    def __enter__(self):
        self.rt = ctypes.CDLL("libamdhip64.so.7")
        self.rt.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
        self.rt.hipFree.argtypes = [ctypes.c_void_p]
        self.blocks = []
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert self.rt.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        if free.value > 512 * MIB:
            self.take(free.value - 256 * MIB)
        while self.take(40 * MIB):
            pass
        return self

    def take(self, size):
        p = ctypes.c_void_p()
        if self.rt.hipMalloc(ctypes.byref(p), size) != 0:
            self.rt.hipGetLastError()
            return False
        self.blocks.append(p)
        return True

    def __exit__(self, *exc):
        for p in self.blocks:
            self.rt.hipFree(p)


def test_one_launch_falls_back_without_memory():
    print("[gpu] out of device memory", flush=True)
    eng = ch.Engine(0)
    try:
        flat = ch.lower(inverter())
        s = eng.load(flat)
        names = ["MN.vth", "CL"]
        n_out = 50 * MIB // (8 * s.n)
        n_sens = 60 * MIB // (8 * s.n * 3)

        def tran(kern):
            return s.tran(ch.grid_options((0.0, 1e-10), n_out=n_out, batch_kernel=kern))

        def sens(kern, n=n_sens):
            return s.tran_sens(ch.grid_options((0.0, 1e-10), n_out=n, batch_kernel=kern), names)

        ref, (ref_s, ref_g) = tran(L.BATCH_KERNEL_GLOBAL), sens(L.BATCH_KERNEL_GLOBAL)
        sens(L.BATCH_KERNEL_AUTO, 3)
        dc = s.dcop()
        with _Fill() as fill:
            assert not fill.take(50 * MIB)
            print("[gpu] filled", flush=True)
            a = tran(L.BATCH_KERNEL_AUTO)
            assert a.retcode == "Success" and np.array_equal(a.wave, ref.wave)
            b, g = sens(L.BATCH_KERNEL_AUTO)
            assert b.retcode == "Success" and np.array_equal(b.wave, ref_s.wave) and np.array_equal(g, ref_g)
            with pytest.raises(ch.CedarHIPError) as e:
                tran(L.BATCH_KERNEL_LDS)
            assert e.value.code == L.CS_E_OOM
            assert np.array_equal(s.dcop().u, dc.u)   # small calls go on
        c = tran(L.BATCH_KERNEL_LDS)
        assert c.retcode == "Success" and np.all(np.abs(c.wave - ref.wave) <= 1e-6 * np.abs(ref.wave) + 1e-9)
    finally:
        eng.close()
