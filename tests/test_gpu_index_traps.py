"""FP32 dsmc_index_atoms where the last move removed atoms in a context of
several traps: the removed atoms still hold slots, and every atom keeps its
trap.  What is observed per trap does not change by indexing, and a step call
by call, with the index, is bitwise that of dsmc_step."""
import numpy as np
import pytest

from cudadsmc_amd import Simulation, _abi, configs

pytestmark = pytest.mark.gpu

FIELDS = [_abi.FIELD_ATOM_ID, _abi.FIELD_POS, _abi.FIELD_VEL, _abi.FIELD_CELL_ID, _abi.FIELD_TRAP_START,
          _abi.FIELD_SIGVRMAX, _abi.FIELD_EVAP_POS]


def _observed(sim):
    return [(o.n_alive, o.ek, o.ep, tuple(o.v2)) for o in sim.observe()]


@pytest.mark.parametrize("sizes", [[700, 1, 2048, 0, 3000, 65], [9000, 0, 25000, 300], [5000] * 3])
@pytest.mark.parametrize("sort_mode", ["incremental", "full"])
@pytest.mark.parametrize("use_graph", [True, False])
def test_index_keeps_traps(sizes, sort_mode, use_graph):
    traps = []
    for k, n in enumerate(sizes):
        t = configs.quadrupole_trap(n, 4 + k, T=(20 + 5 * k) * 1e-6, n_real=1e9)
        t.eta_start = t.eta_end = 4.0
        t.T_cut = t.T
        traps.append(t)
    run = configs.Run(traps=traps, precision="fp32", energy_cut=True, dt=1e-5, seed=6, sort_mode=sort_mode,
                      use_graph=use_graph)
    with Simulation(run) as a, Simulation(run) as b:
        a.init_distribution()
        b.init_distribution()
        for steps in (1, 5, 2):
            a.step(steps)
            b.step(steps)
            before = _observed(a)
            start, key = a.copy_out(_abi.FIELD_TRAP_START), a.copy_out(_abi.FIELD_CELL_ID)
            a.index_atoms()
            a.index_atoms()
            assert _observed(a) == before
            np.testing.assert_array_equal(a.copy_out(_abi.FIELD_TRAP_START), start)
            np.testing.assert_array_equal(a.copy_out(_abi.FIELD_CELL_ID), key)
            a.sort_arrays()
            a.build_cell_table()
            a.collide()
            a.move_atoms()
            b.step(1)
            for f in FIELDS:
                np.testing.assert_array_equal(a.copy_out(f), b.copy_out(f), err_msg=f"field {f}")
        assert 0 < a.info().n_alive < sum(sizes)
