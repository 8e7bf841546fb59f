"""The collide's cell list (a lane holds eight consecutive sorted slots, a wave
512) where cells and the alive atoms end at, before and after the ends of
lanes and chunks: the split step against the fused step, which lists its cells
slot by slot.  Both run the same trials, so the states are bitwise equal."""
import numpy as np
import pytest

from cudadsmc_amd import Simulation, _abi, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 7, 8, 9, 511, 512, 513, 1025, 2050])
@pytest.mark.parametrize("nc", [1, 3, 9])
def test_cells_across_lanes_and_chunks(n, nc, monkeypatch):
    out = {}
    for fused in ("0", "1"):
        monkeypatch.setenv("DSMC_STEP_FUSED", fused)
        run = configs.box_thermalise("fp32", n, nc).with_(use_graph=False, dt=2e-6)
        run.traps[0].n_real = 2.5e12   # n sigma <v_r> dt = 0.2 collisions per atom and step
        with Simulation(run) as sim:
            sim.init_distribution()
            sim.step(6)
            out[fused] = [sim.copy_out(f) for f in (_abi.FIELD_POS, _abi.FIELD_VEL, _abi.FIELD_ATOM_ID,
                                                    _abi.FIELD_SIGVRMAX)]
            out[fused].append(sim.obs_log()["collisions"].copy())
    if n > 500:
        assert out["0"][4].sum() > 20
    for a, b in zip(out["0"], out["1"]):
        np.testing.assert_array_equal(a, b)
