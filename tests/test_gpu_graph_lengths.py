"""Steps replayed from the captured pair of steps, from the long graph of eight
pairs and from both, against the same steps launched one by one, bitwise after
every call: calls below, at and above one pair, eight pairs and the number of
pairs from which the long graph is used, odd ones (which leave the buffers the
other way round), reads and single steps in between, and a re-initialised
context; with and without removed atoms, with the re-sort in the finalize's
launch and outside it."""
import numpy as np
import pytest

from cudadsmc_amd import Simulation, _abi, configs

pytestmark = pytest.mark.gpu

FIELDS = [_abi.FIELD_ATOM_ID, _abi.FIELD_POS, _abi.FIELD_VEL, _abi.FIELD_CELL_ID, _abi.FIELD_PERM,
          _abi.FIELD_SIGVRMAX]
CALLS = [1, 2, 14, 16, 15, 17, 64, 1, 33, 130, 3, 62, 16]


@pytest.mark.parametrize("n", [500, 40000])
@pytest.mark.parametrize("precision,lpc,cut", [("fp32", 1, False), ("fp32", 1, True), ("fp64", 1, True),
                                               ("fp64", 3, False), ("fp64", 17, True)])
def test_replayed_steps_equal_launched_steps(n, precision, lpc, cut):
    trap = configs.quadrupole_trap(n, 9, n_real=1e9)
    if cut:
        trap.eta_start, trap.eta_end, trap.T_cut, trap.eta_steps = 7.0, 4.0, trap.T, 300
    run = configs.Run(traps=[trap], precision=precision, energy_cut=cut, lpc=lpc, dt=1e-6, seed=11)
    with Simulation(run.with_(use_graph=True)) as a, Simulation(run.with_(use_graph=False)) as b:
        for again in range(2):
            a.init_distribution()
            b.init_distribution()
            for k, steps in enumerate(CALLS if again == 0 else [200, 40]):
                steps *= lpc
                a.step(steps)
                b.step(steps)
                if k % 3 == 1:
                    continue
                for f in FIELDS:
                    np.testing.assert_array_equal(a.copy_out(f), b.copy_out(f), err_msg=f"field {f}, call {k}")
                la, lb = a.obs_log(), b.obs_log()
                for f in la.dtype.names:
                    np.testing.assert_array_equal(la[f], lb[f], err_msg=f)


def test_runs_with_reads_between():
    """Reads of a run with losses swap the state's buffers: two captured states
    in turn, and a third (an odd number of steps) in place of the older."""
    trap = configs.quadrupole_trap(3000, 9, n_real=1e9)
    trap.eta_start, trap.eta_end, trap.T_cut, trap.eta_steps = 6.0, 3.0, trap.T, 2000
    run = configs.Run(traps=[trap], precision="fp64", energy_cut=True, dt=1e-6, seed=5)
    with Simulation(run.with_(use_graph=True)) as a, Simulation(run.with_(use_graph=False)) as b:
        a.init_distribution()
        b.init_distribution()
        for steps in [40, 40, 40, 80, 80, 41, 40, 40, 43, 90, 90, 90, 90]:
            a.step(steps)
            b.step(steps)
            for f in FIELDS:
                np.testing.assert_array_equal(a.copy_out(f), b.copy_out(f))
        assert a.info().n_alive == b.info().n_alive < 3000


@pytest.mark.parametrize("sort_mode", ["full", "incremental"])
@pytest.mark.parametrize("precision,cut", [("fp32", False), ("fp32", True), ("fp64", True)])
def test_a_new_run_replays_the_last_ones_steps(precision, cut, sort_mode):
    """A re-initialised context may begin with a graph of its earlier run: what
    the steps leave (which order is current, whether atoms were removed) is
    then that of the new run."""
    n = 777
    trap = configs.quadrupole_trap(n, 9, n_real=1e9)
    if cut:
        trap.eta_start = trap.eta_end = 4.0
        trap.T_cut = trap.T
    run = configs.Run(traps=[trap], precision=precision, energy_cut=cut, dt=1e-6, seed=4, sort_mode=sort_mode)
    rng = np.random.default_rng(3)
    pos = rng.normal(0.0, 0.2, (n, 3)) * np.array(trap.half_width)
    vel = rng.normal(0.0, 0.05, (n, 3))
    with Simulation(run.with_(use_graph=True)) as a, Simulation(run.with_(use_graph=False)) as b:
        for sim in (a, b):
            sim.init_distribution()
            sim.step(80)
            if precision == "fp32":   # an odd number of sorts before the new run
                sim.sort_arrays()
                sim.collide()
                sim.move_atoms()
        for steps in (70, 2, 1, 40):
            for sim in (a, b):
                sim.set_state(pos, vel)
                sim.step(steps)
            assert a.info().n_alive == b.info().n_alive
            assert not cut or a.info().n_alive < n
            for f in FIELDS:
                np.testing.assert_array_equal(a.copy_out(f), b.copy_out(f), err_msg=f"field {f}")
            oa, ob = a.observe()[0], b.observe()[0]
            assert (oa.n_alive, oa.ek, oa.ep) == (ob.n_alive, ob.ek, ob.ep)
