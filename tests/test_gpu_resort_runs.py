"""FP64 steps called one after the other without a read in between, at the
capacity (32768) up to which the whole re-sort runs beside the finalize: with
losses, removed atoms then still hold slots when the next call begins (a read
would drop them).  Bitwise equal to the same steps call by call, with graphs
and without, in calls that end inside a collision step and at its end."""
import numpy as np
import pytest

from cudadsmc_amd import Simulation, _abi, configs

pytestmark = pytest.mark.gpu

FIELDS = [_abi.FIELD_ATOM_ID, _abi.FIELD_POS, _abi.FIELD_VEL, _abi.FIELD_ACC, _abi.FIELD_CELL_ID, _abi.FIELD_PERM,
          _abi.FIELD_SIGVRMAX, _abi.FIELD_CELL_COUNT, _abi.FIELD_COLLISION_COUNT]


@pytest.mark.parametrize("use_graph", [False, True])
@pytest.mark.parametrize("n", [1000, 32767, 32768, 32769, 36865])
@pytest.mark.parametrize("dt,cut,lpc", [(1e-6, True, 1), (1e-6, True, 3), (1e-4, True, 1), (1e-4, False, 2)])
def test_calls_without_a_read_between(n, dt, cut, lpc, use_graph):
    trap = configs.quadrupole_trap(n, 12, n_real=1e9)
    if cut:
        trap.eta_start = trap.eta_end = 5.0
        trap.T_cut = trap.T
    run = configs.Run(traps=[trap], precision="fp64", energy_cut=cut, dt=dt, seed=3, lpc=lpc, use_graph=use_graph)
    with Simulation(run) as a, Simulation(run) as b:
        a.init_distribution()
        b.init_distribution()
        calls = [lpc, 2 * lpc, 5 * lpc, 1, 4 * lpc, 7 * lpc - 1, 2 * lpc]
        for steps in calls:
            a.step(steps)
        for s in range(sum(calls)):
            if s % lpc == 0:
                b.index_atoms()
                b.sort_arrays()
                b.build_cell_table()
                b.collide()
            b.move_atoms()
            if cut:
                b.evaporation_tag()
                b.compact()
        assert a.info().n_alive == b.info().n_alive
        assert not cut or a.info().n_alive < n
        assert a.obs_log()["collisions"].sum() > 0
        for f in FIELDS:
            np.testing.assert_array_equal(a.copy_out(f), b.copy_out(f), err_msg=f"field {f}")
