"""A neighbour list that overflows keeps the state: the step or run reports it
and the particles are where they were at the start of that step, however many
rows overflow and wherever in their stencil.  The lists are a fraction of the
neighbours, so that most rows stop before they reach the particle's own cell and
the overflowed rows count more faces than complete lists could have."""
import numpy as np
import pytest

from cases import jitter3d, jitter3d_open, kh_lattice, kh_open
from meshlesshydro_amd import learned as L
from meshlesshydro_amd._abi import (MLH_ERR_NEIGHBOUR_OVERFLOW, MLH_FP32, MLH_ORDER_CALLER,
                                    MLH_SEED_LEARNED)

pytestmark = pytest.mark.gpu

CASES = {
    "open2d": (kh_open, dict(max_interactions=6)),
    "open3d": (jitter3d_open, dict(max_interactions=6)),
    # image lists shorter than half the real ones
    "box2d": (kh_lattice, dict(n=40, max_interactions=6, max_ghost_interactions=1)),
    "box3d": (jitter3d, dict(max_interactions=12, max_ghost_interactions=1)),
}
MODES = {
    "fp64": {},
    "fp32": dict(precision=MLH_FP32),
    "fp32_learned": dict(precision=MLH_FP32, riemann_seed=MLH_SEED_LEARNED),
    "caller": dict(work_order=MLH_ORDER_CALLER),
    "both_sides": dict(enforce_flux_sym=0),
}


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("call", ["step", "run"])
def test_state_kept(call, case, mode, hip):
    make, kw = CASES[case]
    p, s = make(debug_level=0, **kw, **MODES[mode])
    print(f"\n[overflow state {call}/{case}/{mode}]", flush=True)
    sim = hip.Simulation(p, s)
    if mode.endswith("learned"):
        sim.mlp_set_params(L.init_params(1))
    for _ in range(2):
        with pytest.raises(hip.MLHError) as e:
            sim.step() if call == "step" else sim.run(3)
        assert e.value.status == MLH_ERR_NEIGHBOUR_OVERFLOW
        got = sim.state()
        for k in got:
            assert np.array_equal(got[k], s[k]), k
    sim.close()
