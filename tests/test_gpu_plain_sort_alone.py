"""FP64 dsmc_sort_arrays on its own after dsmc_step: the keys that it sorts are
those which the step's index and sort leave, as after the same steps call by
call, whatever the number of radix passes (one and three leave the keys of the
slots before the sort, two the sorted ones), in the middle of a collision step
and at its end, with removed atoms and without, launched and replayed."""
import numpy as np
import pytest

from cudadsmc_amd import Simulation, _abi, configs

pytestmark = pytest.mark.gpu

FIELDS = [_abi.FIELD_PERM, _abi.FIELD_CELL_ID, _abi.FIELD_ATOM_ID, _abi.FIELD_POS, _abi.FIELD_VEL,
          _abi.FIELD_COLLISION_COUNT]


@pytest.mark.parametrize("n,nc,passes", [(3000, 5, 1), (3000, 12, 2), (70000, 45, 3)])
@pytest.mark.parametrize("lpc,cut", [(1, False), (1, True), (3, True), (3, False)])
@pytest.mark.parametrize("steps", [1, 4, 30, 72])
def test_sort_after_steps(n, nc, passes, lpc, cut, steps):
    trap = configs.quadrupole_trap(n, nc, n_real=1e9)
    if cut:
        trap.eta_start = trap.eta_end = 5.0
        trap.T_cut = trap.T
    run = configs.Run(traps=[trap], precision="fp64", energy_cut=cut, dt=1e-5, seed=7, lpc=lpc)
    with Simulation(run) as a, Simulation(run) as b:
        assert a.info().radix_passes == passes
        a.init_distribution()
        b.init_distribution()
        a.step(steps)
        for s in range(steps):
            if s % lpc == 0:
                b.index_atoms()
                b.sort_arrays()
                b.build_cell_table()
                b.collide()
            b.move_atoms()
            if cut:
                b.evaporation_tag()
                b.compact()
        for sim in (a, b):
            sim.sort_arrays()
            sim.build_cell_table()
            sim.collide()
        for f in FIELDS:
            np.testing.assert_array_equal(a.copy_out(f), b.copy_out(f), err_msg=f"field {f}")
        for sim in (a, b):   # once more, and on with steps
            sim.sort_arrays()
            sim.step(2 * lpc - steps % lpc)
        for f in FIELDS[2:5]:
            np.testing.assert_array_equal(a.copy_out(f), b.copy_out(f), err_msg=f"field {f}")
