"""The incremental re-sort where tiles (2048 slots), first-phase blocks (4096)
and buckets (512 movers in LDS, 1024 in the room) begin and end: whole runs
bitwise equal to those that radix-sort every key, with few and with nearly all
atoms changing cell, with removed atoms and without."""
import numpy as np
import pytest

from cudadsmc_amd import Simulation, _abi, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 2047, 2048, 2049, 4095, 4096, 4097, 6145])
@pytest.mark.parametrize("dt,cut", [(1e-6, False), (1e-6, True), (1e-4, False), (1e-4, True)])
def test_incremental_equals_full(n, dt, cut):
    trap = configs.quadrupole_trap(n, 12)
    if cut:
        trap.eta_start, trap.eta_end, trap.T_cut, trap.eta_steps = 7.0, 4.0, trap.T, 20
    out = {}
    for mode in ("incremental", "full"):
        run = configs.Run(traps=[trap], precision="fp32", energy_cut=cut, dt=dt, seed=3, sort_mode=mode)
        with Simulation(run) as sim:
            sim.init_distribution()
            for steps in (1, 2, 9, 20):
                sim.step(steps)
                out.setdefault(mode, []).extend(
                    sim.copy_out(f) for f in (_abi.FIELD_ATOM_ID, _abi.FIELD_POS, _abi.FIELD_VEL, _abi.FIELD_CELL_ID,
                                              _abi.FIELD_PERM))
            # the order itself: cells ascending, slots ascending within a cell
            sim.sort_arrays()
            key, perm = sim.copy_out(_abi.FIELD_CELL_ID), sim.copy_out(_abi.FIELD_PERM)
            assert (np.lexsort((perm, key)) == np.arange(len(key))).all()
            out[mode] += [key, perm]
    for a, b in zip(out["incremental"], out["full"]):
        np.testing.assert_array_equal(a, b)
