"""The fused step (DSMC_STEP_FUSED=1) where cells lie across the boundaries
between its waves' spans: both waves run such a cell's trials from the sigma
v_r,max that the step began with, and the value that the trials raise is stored
after them, so the states are bitwise those of the split step in every run.
Many spans, dense cells and a sigma v_r,max that grows in every step."""
import numpy as np
import pytest

from cudadsmc_amd import Simulation, _abi, configs

pytestmark = pytest.mark.gpu

FIELDS = [_abi.FIELD_POS, _abi.FIELD_VEL, _abi.FIELD_ATOM_ID, _abi.FIELD_SIGVRMAX]


@pytest.mark.parametrize("n,traps,nc,block", [(757, 520, 5, 0), (757, 520, 5, 64), (757, 520, 5, 1024),
                                              (400000, 1, 36, 0), (65, 1, 2, 64), (129, 1, 3, 128)])
def test_fused_step_with_growing_sigvrmax(n, traps, nc, block, monkeypatch):
    out = []
    for fused in ("0", "1", "1", "1"):
        monkeypatch.setenv("DSMC_STEP_FUSED", fused)
        run = configs.box_thermalise("fp32", n, nc).with_(dt=2e-6, use_graph=False, block_size=block)
        box = run.traps[0]
        box.n_real = 2.5e12   # n sigma <v_r> dt = 0.2 collisions per atom and step
        box.T_axis = (4e-6, 40e-6, 400e-6)
        run = run.with_(traps=[box] * traps)
        with Simulation(run) as sim:
            sim.init_distribution()
            first = sim.copy_out(_abi.FIELD_SIGVRMAX)
            sim.step(8)
            out.append([sim.copy_out(f) for f in FIELDS] + [sim.obs_log()["collisions"].copy()])
        assert n * traps < 1000 or (out[-1][3] > first).sum() > 100
        for a, b in zip(out[0], out[-1]):
            np.testing.assert_array_equal(a, b)
