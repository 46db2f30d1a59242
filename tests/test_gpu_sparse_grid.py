"""Sparse clouds without periodic boundaries: many more search cells than
particles."""
import numpy as np
import pytest

from cases import relerr
from meshlesshydro_amd._abi import MLH_ABS_FABS, default_params

pytestmark = pytest.mark.gpu

H, CELLS = 0.02, 215


def cloud(n, seed=5):
    """clumps of 50 particles within about a kernel, drawn over CELLS kernels
    per axis, two of them at opposite corners"""
    rng = np.random.default_rng(seed)
    c = rng.uniform(0.0, CELLS * H, (3, n // 50))
    c[:, 0], c[:, 1] = 0.0, CELLS * H
    x = np.repeat(c, 50, axis=1) + rng.uniform(0.0, 1.2 * H, (3, n))
    v = rng.uniform(-0.1, 0.1, (3, n))
    s = dict(x=x[0], y=x[1], z=x[2], vx=v[0], vy=v[1], vz=v[2], m=np.full(n, 1.0 / n), u=rng.uniform(1.0, 1.2, n))
    return default_params(dim=3, periodic=0, kernel_size=H, debug_level=0, limiter_abs=MLH_ABS_FABS), s


@pytest.mark.parametrize("n", [600, 20000])
def test_rows_and_density(n, hip, oracle_mod):
    p, s = cloud(n)
    print(f"\n[sparse cloud {n}]", flush=True)
    sim, orc = hip.Simulation(p, s), oracle_mod.Oracle(p, s)
    for _ in range(2):
        sim.neighbours()
    orc.neighbours()
    (gn, gg, gl), (on, og, ol) = sim.get_neighbours(), orc.get_neighbours()
    assert np.array_equal(gn, on) and np.array_equal(gg, og)
    mask = np.arange(gl.shape[1])[None, :] < (gn + gg)[:, None]
    assert np.array_equal(np.where(mask, gl, 0), np.where(mask, ol, 0))
    sim.density()
    orc.density()
    for a, b in zip(sim.get_density(), orc.get_density()):
        assert relerr(a, b) < 1e-10
    sim.close()


def test_few_particles_search_as_fast_as_many(hip):
    """Clearing the cells is the chip's work, however few the particles: the
    search of 600 takes no longer than 1.5 times that of 20000 on the same
    grid."""
    ms = []
    for n in (600, 20000):
        p, s = cloud(n)
        sim = hip.Simulation(p, s)
        t = []
        for _ in range(6):
            sim.upload(s)
            sim.step(dt_fixed=1e-9)
            t.append(float(sim.timings()[0]))
        ms.append(min(t))
        print(f"\n[sparse search {n}] {ms[-1]} ms", flush=True)
        sim.close()
    assert ms[0] < 1.5 * ms[1], ms
