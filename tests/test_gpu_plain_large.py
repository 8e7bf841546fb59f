"""FP64 contexts beyond the incremental re-sort's limit (2^24 atoms), whose
steps radix-sort the cell keys that the previous step left: replayed steps
against launched ones, bitwise, where the keys are not those of the state when
a call begins -- the first call of a new context, with atoms removed from the
start, and short calls that replay a graph of an earlier run after a new
distribution, a new state and a single call."""
import numpy as np
import pytest

from cudadsmc_amd import Simulation, _abi, configs

pytestmark = pytest.mark.gpu

N = 1 << 24


def _run(cut, use_graph):
    trap = configs.quadrupole_trap(N, 160, n_real=1e9)
    if cut:
        trap.eta_start = trap.eta_end = 6.0
        trap.T_cut = trap.T
    return configs.Run(traps=[trap], precision="fp64", energy_cut=cut, dt=1e-5, seed=2, use_graph=use_graph)


def _new_distribution(sim):
    sim.init_distribution()


def _new_state(sim):
    rng = np.random.default_rng(1)
    hw = np.array(sim.run.traps[0].half_width)
    sim.set_state(rng.normal(0.0, 0.2, (N, 3)) * hw, rng.normal(0.0, 0.05, (N, 3)))


def _single_call(sim):
    sim.move_atoms()


@pytest.mark.parametrize("cut", [False, True])
@pytest.mark.parametrize("first,between,steps", [(6, None, 0), (82, _new_distribution, 2), (82, _single_call, 2),
                                                 (2, _new_state, 7)])
def test_replayed_steps_equal_launched_steps(cut, first, between, steps):
    out = {}
    for use_graph in (True, False):
        with Simulation(_run(cut, use_graph)) as sim:
            sim.init_distribution()
            sim.step(first)
            if between:
                between(sim)
                sim.step(steps)
            print(f"graph {use_graph}: {sim.info().n_alive} alive", flush=True)
            out[use_graph] = [sim.info().n_alive, sim.obs_log()["collisions"].copy()]
            out[use_graph] += [sim.copy_out(f) for f in (_abi.FIELD_ATOM_ID, _abi.FIELD_VEL, _abi.FIELD_SIGVRMAX)]
    assert (out[True][0] < N) == cut and out[True][1].sum() > 0
    for a, b in zip(out[True], out[False]):
        assert np.array_equal(a, b)
