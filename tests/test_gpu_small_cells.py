"""The cell list of a small problem is built in one block, that of a larger
one in passes over the chip: neighbour rows and densities on both sides of the
sizes where the rounds and the route change, against the oracle."""
import numpy as np
import pytest

from cases import relerr
from meshlesshydro_amd._abi import MLH_ABS_FABS, default_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("N", [65, 1023, 1025, 16384, 16385])
def test_rows_and_density(hip, oracle_mod, dim, N):
    rng = np.random.default_rng(N + dim)
    s = {k: rng.random(N) for k in ("x", "y", "z")[:dim]}
    for k in ("vx", "vy", "vz")[:dim]:
        s[k] = rng.uniform(-0.1, 0.1, N)
    s["m"], s["u"] = np.full(N, 1.0 / N), rng.uniform(1.0, 1.2, N)
    # 24 neighbours in the mean; a quarter of the box at most
    vol = 24.0 / N
    h = min(0.25, (vol / np.pi) ** 0.5 if dim == 2 else (vol * 0.75 / np.pi) ** (1 / 3))
    p = default_params(kernel_size=h, dim=dim, limiter_abs=MLH_ABS_FABS)
    print(f"\n[small cells {dim}D N={N}] h={h}", flush=True)
    sim, orc = hip.Simulation(p, s), oracle_mod.Oracle(p, s)
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
