"""More than 2^26 particles, where an image's sort word no longer holds its
parent: the images at the faces of a periodic lattice, by the volume that the
densities sum up to, and the search's time."""
import time

import numpy as np
import pytest

from meshlesshydro_amd._abi import MLH_FP32, MLH_FP64, default_params

pytestmark = pytest.mark.gpu


def lattice(n, dim):
    c, z = (np.arange(n) + 0.5) / n, np.zeros(n ** dim)
    x = [np.tile(np.repeat(c, n ** (dim - 1 - a)), n ** a) for a in range(dim)]
    s = dict(zip(("x", "y", "z"), x), m=np.full(n ** dim, 1.0 / n ** dim), u=np.ones(n ** dim))
    return s | {k: z for k in ("vx", "vy", "vz")[:dim]}


def kernel_2d(r, h):
    """the cubic spline of support h: 10 / (7 pi (h/2)^2) times the piecewise cubic"""
    q = r / (h / 2.0)
    w = np.where(q < 1.0, 1.0 - 1.5 * q ** 2 * (1.0 - q / 2.0), np.where(q < 2.0, 0.25 * (2.0 - q) ** 3, 0.0))
    return 10.0 / (7.0 * np.pi * (h / 2.0) ** 2) * w


def test_lattice_volume(hip):
    n = 8200
    assert n * n > 1 << 26
    dx, h = 1.0 / n, 2.2 / n
    s = lattice(n, 2)
    p = default_params(kernel_size=h, max_interactions=16, max_ghost_interactions=12, debug_level=0,
                       precision=MLH_FP64)
    print(f"\n[{n}^2 particles]", flush=True)
    sim = hip.Simulation(p, s)
    sim.neighbours()
    sim.density()
    d = sim.diag()
    volume = sim.conserved()[0]
    sim.close()
    # sqrt(5) > 2.2: twelve neighbours; a corner particle has three of them inside
    # at distance 1 and sqrt 2, two at distance 2, and seven images
    assert d["max_neighbours"] == 12 and d["max_ghost_neighbours"] == 7
    k = np.arange(-3, 4)
    r = dx * np.hypot(*np.meshgrid(k, k))
    omega = np.sum(kernel_2d(r[r < h], h))
    # one particle's missing image at distance 1 would change it by 2e-9, at sqrt 2
    # by 5e-10; coordinates are exact to 1e-12 of dx
    assert abs(volume * omega / (n * n) - 1.0) < 5e-11, volume * omega / (n * n) - 1.0


def test_search_time(hip):
    """407^3 particles search as fast as 406^3, which lie below 2^26: within 1.1
    (1.01 times as many)."""
    ms = []
    for n in (406, 407):
        p = default_params(dim=3, kernel_size=2.05 / n, max_interactions=40, max_ghost_interactions=40, debug_level=0,
                           precision=MLH_FP32)
        print(f"\n[{n}^3 particles]", flush=True)
        sim = hip.Simulation(p, lattice(n, 3))
        t = []
        for _ in range(10):
            t0 = time.perf_counter()
            sim.neighbours()
            t.append(1e3 * (time.perf_counter() - t0))
        ms.append(min(t))
        print(f"[search {n}^3] {ms[-1]} ms", flush=True)
        sim.close()
    assert ms[1] < 1.1 * ms[0], ms
