"""The FP64 form's whole step (dsmc_step) against the same loop call by call
(index, sort, table, collide, then move, tag and compact per motion step): the
state, the cell table and what the last calls left are bitwise equal, at the
edges of blocks and tiles, with calls that end inside a collision step, with
removed atoms, and with more motion substeps than one launch takes."""
import numpy as np
import pytest

from cudadsmc_amd import Simulation, _abi, configs

pytestmark = pytest.mark.gpu

FIELDS = [_abi.FIELD_POS, _abi.FIELD_VEL, _abi.FIELD_ACC, _abi.FIELD_ATOM_ID, _abi.FIELD_CELL_ID,
          _abi.FIELD_PERM, _abi.FIELD_EVAP_POS, _abi.FIELD_EVAP_VEL, _abi.FIELD_CELL_START_END,
          _abi.FIELD_CELL_COUNT, _abi.FIELD_CELL_PREFIX, _abi.FIELD_SIGVRMAX, _abi.FIELD_COLLISION_COUNT]


def _by_calls(sim, steps, at):
    for s in range(at, at + steps):
        if s % sim.run.lpc == 0:
            sim.index_atoms()
            sim.sort_arrays()
            sim.build_cell_table()
            sim.collide()
        sim.move_atoms()
        if sim.run.energy_cut:
            sim.evaporation_tag()
            sim.compact()


@pytest.mark.parametrize("n", [1, 255, 257, 2049, 5000])
@pytest.mark.parametrize("lpc,kind,cut", [(1, "quadrupole", False), (1, "quadrupole", True), (3, "box", False),
                                          (17, "quadrupole", True), (2, "ip", True)])
def test_step_equals_calls(n, lpc, kind, cut):
    if kind == "box":
        run = configs.box_thermalise("fp64", n, 5)
        run.traps[0].n_real = 2e12
    elif kind == "ip":
        t = configs.reference(20, n).traps[0]
        run = configs.Run(traps=[t])
    else:
        run = configs.Run(traps=[configs.quadrupole_trap(n, 9, n_real=1e9)])
    t = run.traps[0]
    if cut:   # constant, so that it does not matter when it is read
        t.eta_start = t.eta_end = 5.0
        t.T_cut = t.T
    run = run.with_(energy_cut=cut, lpc=lpc, dt=1e-6, seed=n)
    fields = FIELDS + ([_abi.FIELD_EVAP_TAG] if cut else [])
    with Simulation(run) as a, Simulation(run) as b:
        a.init_distribution()
        b.init_distribution()
        at = 0
        # the last calls are long enough to replay the graph
        for steps in (1, 2, 4, 2 * lpc, 1, 5 * lpc + 1, 4 * lpc):
            a.step(steps)
            _by_calls(b, steps, at)
            at += steps
            for f in fields:
                np.testing.assert_array_equal(a.copy_out(f), b.copy_out(f), err_msg=f"field {f} at step {at}")
        ia, ib = a.info(), b.info()
        assert (ia.n_alive, ia.step, ia.collision_steps) == (ib.n_alive, ib.step, ib.collision_steps)
        # and on without a read in between, which lets removed atoms keep their slots
        for steps in (1, lpc, 2, 3 * lpc):
            a.step(steps)
            _by_calls(b, steps, at)
            at += steps
        for f in fields:
            np.testing.assert_array_equal(a.copy_out(f), b.copy_out(f), err_msg=f"field {f} at the end")
        if n > 2000:
            assert not cut or ia.n_alive < n
            assert kind == "ip" or a.obs_log()["collisions"].sum() > 0


@pytest.mark.parametrize("n", [1, 63, 255, 257, 4096, 4097, 20000])
@pytest.mark.parametrize("nc", [1, 4, 7, 20])
def test_cell_table(n, nc):
    """start/end, count and prefix of every cell from the sorted keys: blocks of
    256 cells with more or fewer keys than fit LDS, empty cells, the last block."""
    run = configs.Run(traps=[configs.quadrupole_trap(n, nc)])
    with Simulation(run) as sim:
        sim.init_distribution()
        sim.index_atoms()
        sim.sort_arrays()
        sim.build_cell_table()
        key = sim.copy_out(_abi.FIELD_CELL_ID)
        se, count, prefix = (sim.copy_out(f) for f in (_abi.FIELD_CELL_START_END, _abi.FIELD_CELL_COUNT,
                                                       _abi.FIELD_CELL_PREFIX))
    want = np.bincount(key, minlength=nc ** 3 + 1)
    first = np.concatenate([[0], np.cumsum(want)[:-1]])
    np.testing.assert_array_equal(count, want)
    np.testing.assert_array_equal(prefix, first)
    np.testing.assert_array_equal(se[:, 0], np.where(want > 0, first, -1))
    np.testing.assert_array_equal(se[:, 1], np.where(want > 0, first + want - 1, -1))
