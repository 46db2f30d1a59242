"""Device memory for the fluxes of faces evaluated once per pair: who takes it,
and what is left of the device."""
import ctypes as C
import gc

import numpy as np
import pytest

from cases import jitter3d, relerr
from meshlesshydro_amd import learned as L
from meshlesshydro_amd._abi import MLH_FP32, MLH_FP64, MLH_SEED_LEARNED

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


class Fill:
    """All but `leave` bytes of the free device memory, while in scope."""

    def __init__(self, hip, leave):
        self.bufs = []
        n = free_bytes(hip) - leave
        assert n > 0
        while n > 0:
            self.bufs.append(hip.DeviceBuffer(min(n, 16 << 30), np.uint8))
            n -= 16 << 30

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        for b in self.bufs:
            b.free()


def used_by(hip, p, s):
    """(device memory of a context for state s, free memory with it)"""
    before = free_bytes(hip)
    sim = hip.Simulation(p, s)
    after = free_bytes(hip)
    sim.close()
    return before - after, after


def test_slots_leave_the_device_to_others(hip):
    """Slots take a quarter at most of what is free without them."""
    p, s = jitter3d(100, debug_level=0)
    gc.collect()
    with Fill(hip, 6 << 30):
        with_slots, free = used_by(hip, p, s)
        p.enforce_flux_sym = 0
        without, _ = used_by(hip, p, s)
        slots = with_slots - without
        print(f"\n[slots] {slots >> 20} MiB of {(free + slots) >> 20}", flush=True)
        # 40 slots of 40 bytes a particle would be 1526 MiB
        assert 0 < slots <= (free + slots) // 4 + (64 << 20)


def test_slots_make_room_for_the_face_arrays(hip):
    """A stage whose arrays the slots leave no room for gets the slots' memory,
    and the context goes on without them: the same bits."""
    p, s = jitter3d(100, debug_level=0, max_interactions=96, max_ghost_interactions=64)
    arrays = s["x"].size * (96 + 64) * 8 * 21
    slots = s["x"].size * 40 * 40
    ref = hip.Simulation(p, s)
    sim = hip.Simulation(p, s)
    with Fill(hip, arrays - 3 * slots // 4):
        out = []
        for q in (ref, sim):
            q.neighbours()
            q.density()
            dt = q.timestep()
            q.gradients()
            if q is sim:
                q.effective_faces()
            q.upload(s)
            q.run(2)
            out.append((dt, q.state()))
        sim.close()
    ref.close()
    (dt0, s0), (dt1, s1) = out
    assert dt0 == dt1
    for k in s0:
        assert np.array_equal(s0[k], s1[k]), k


def test_long_rows_have_slots_from_the_second_step(hip):
    """Rows of 125 entries outgrow the slots a context starts with: only the first
    step of a fresh context's run evaluates its faces from both sides (1.4 times
    the face stage of the pairs), so the run is within 1.2 of a second one."""
    p, s = jitter3d(56, kernel_size=3.1 / 56, debug_level=0, max_interactions=200, max_ghost_interactions=200)
    sim = hip.Simulation(p, s)
    ms, out = [], []
    for k in range(2):
        print(f"\n[long rows] run {k}", flush=True)
        sim.upload(s)
        dts = sim.run(8)
        ms.append(float(sim.timings()[3]))
        out.append((dts, sim.state()))
    sim.close()
    assert ms[0] < 1.2 * ms[1], ms
    assert np.array_equal(out[0][0], out[1][0])
    for k in out[0][1]:
        assert np.array_equal(out[0][1][k], out[1][1][k]), k


@pytest.mark.parametrize("seed", ["standard", "learned"])
def test_very_long_rows_are_no_slower_in_pairs(seed, hip):
    """Rows of 600 entries, where looking a mirrored entry up costs more than the
    evaluation it saves (1.5 times the face stage): the faces are evaluated
    from both sides, as without flux symmetry."""
    p, s = jitter3d(48, kernel_size=5.24 / 48, debug_level=0, max_interactions=1000, max_ghost_interactions=1000,
                    precision=MLH_FP32)
    if seed == "learned":
        p.riemann_seed = MLH_SEED_LEARNED
    ms = []
    for sym in (1, 0):
        p.enforce_flux_sym = sym
        sim = hip.Simulation(p, s)
        if seed == "learned":
            sim.mlp_set_params(L.init_params(1))
        for k in range(3):
            print(f"\n[very long rows {seed}] symmetry {sym} run {k}", flush=True)
            sim.upload(s)
            sim.run(2)
        ms.append(float(sim.timings()[3]))
        sim.close()
    assert ms[0] < 1.2 * ms[1], ms
