"""The batched Riemann solver gives a face the same bits whatever the number of
blocks its batch is dealt to: batches on both sides of the lines between the
launches (2^18 and 2^22 faces), the shorter ones the first faces of the longer."""
import numpy as np
import pytest

from meshlesshydro_amd import ics, learned
from meshlesshydro_amd._abi import (MLH_FP32, MLH_FP64, MLH_SEED_LEARNED, MLH_SEED_STANDARD, default_params)

pytestmark = pytest.mark.gpu
G = 5.0 / 3.0


@pytest.mark.parametrize("precision", [MLH_FP64, MLH_FP32])
@pytest.mark.parametrize("seed", [MLH_SEED_STANDARD, MLH_SEED_LEARNED])
def test_faces_do_not_depend_on_the_blocks(hip, seed, precision):
    s = np.stack(ics.riemann_states(1 << 16, seed=7))
    s = np.tile(s, (1, 64))
    # near-uniform in every other thousand
    calm = (np.arange(s.shape[1]) // 1000) % 2 == 1
    for q, v in enumerate((1.0, 0.0, 1.0, 1.001, 0.01, 1.01)):
        s[q, calm] = v
    sim = hip.Simulation(default_params(kernel_size=0.1),
                         {k: np.array([0.5]) for k in ("x", "y", "m", "u")} | {k: np.zeros(1) for k in ("vx", "vy")})
    sim.mlp_set_params(learned.init_params(5))
    whole = None
    for n in (1 << 22, (1 << 22) - 1, (1 << 20) + 77, (1 << 18) + 1, 1 << 18):
        print(f"\n[blocks] {n} faces, precision {precision}, seed {seed}", flush=True)
        got = sim.riemann(*s[:, :n], precision=precision, seed=seed)
        whole = whole or got
        for a, b in zip(whole, got):
            np.testing.assert_array_equal(np.asarray(a)[:n], b)
    sim.close()
