"""Device memory for the fluxes of faces evaluated once per pair: who takes it,
and what is left of the device."""
import ctypes as C
import gc

import pytest

from cases import jitter3d, relerr
from meshlesshydro_amd._abi import MLH_FP32, MLH_FP64

pytestmark = pytest.mark.gpu


def free_bytes(hip):
    """free device memory, as the library's runtime sees it"""
    free, total = C.c_size_t(), C.c_size_t()
    f = hip.lib().hipMemGetInfo
    f.restype, f.argtypes = C.c_int, [C.POINTER(C.c_size_t)] * 2
    assert f(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("prec", [MLH_FP64, MLH_FP32])
def test_no_slots_without_flux_symmetry(prec, hip):
    """Above 2^16 particles in 3D no face is shared without flux symmetry, and no
    slots are taken for it."""
    n = 56
    p, s = jitter3d(n, debug_level=0, precision=prec)
    used = {}
    for sym in (1, 0):
        p.enforce_flux_sym = sym
        gc.collect()
        before = free_bytes(hip)
        sim = hip.Simulation(p, s)
        used[sym] = before - free_bytes(hip)
        sim.close()
    slot = 5 * (8 if prec == MLH_FP64 else 4)
    # 40 slots a particle
    assert used[1] - used[0] > 0.9 * 40 * slot * n ** 3


@pytest.mark.parametrize("n", [40, 41])  # 64000 and 68921 particles: either side of 2^16
def test_no_flux_symmetry_vs_oracle(n, hip, oracle_mod):
    p, s = jitter3d(n, debug_level=0, enforce_flux_sym=0, precision=MLH_FP64)
    print(f"\n[no flux symmetry {n}^3]", flush=True)
    sim, orc = hip.Simulation(p, s), oracle_mod.Oracle(p, s)
    dt_o, dt_g = orc.step(), sim.step()
    assert abs(dt_g - dt_o) <= 1e-11 * dt_o
    gs, os_ = sim.state(), orc.state()
    sim.close()
    for k in gs:
        assert relerr(gs[k], os_[k]) < 1e-9, k
