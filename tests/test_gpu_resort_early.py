"""Re-sorts on both sides of the capacity (32768) up to which the whole re-sort
runs beside the finalize and above which it is a first phase and a merge: whole
runs bitwise equal to those that radix-sort every key (FP32) or that are driven
call by call (FP64), at the edges of tiles and blocks, with few and with nearly
all atoms changing cell, with removed atoms and without, for one trap and
several, and with calls in between that read or re-index the state."""
import numpy as np
import pytest

from cudadsmc_amd import Simulation, _abi, configs

pytestmark = pytest.mark.gpu

FIELDS = [_abi.FIELD_ATOM_ID, _abi.FIELD_POS, _abi.FIELD_VEL, _abi.FIELD_CELL_ID, _abi.FIELD_PERM]


def _trap(n, cut, nc=12):
    trap = configs.quadrupole_trap(n, nc)
    if cut:
        trap.eta_start, trap.eta_end, trap.T_cut, trap.eta_steps = 7.0, 4.0, trap.T, 20
    return trap


@pytest.mark.parametrize("sizes", [[32767], [32768], [32769], [34815], [34816], [34817], [36865], [40961],
                                   [2048, 1, 30719], [2048, 1, 30720], [5000, 0, 31000], [700] * 46, [700] * 47])
@pytest.mark.parametrize("dt,cut", [(1e-6, False), (1e-6, True), (1e-4, False), (1e-4, True)])
def test_incremental_equals_full(sizes, dt, cut):
    out = {}
    for mode in ("incremental", "full"):
        run = configs.Run(traps=[_trap(n, cut) for n in sizes], precision="fp32", energy_cut=cut, dt=dt, seed=3,
                          sort_mode=mode)
        with Simulation(run) as sim:
            sim.init_distribution()
            for steps in (1, 2, 9, 20):
                sim.step(steps)
                out.setdefault(mode, []).extend(sim.copy_out(f) for f in FIELDS)
            sim.sort_arrays()   # by calls
            key, perm = sim.copy_out(_abi.FIELD_CELL_ID), sim.copy_out(_abi.FIELD_PERM)
            assert (np.lexsort((perm, key)) == np.arange(len(key))).all()
            sim.collide()
            sim.move_atoms()
            out[mode] += [key, perm, sim.copy_out(_abi.FIELD_VEL)]
            sim.step(4)         # and on from there
            out[mode] += [sim.copy_out(f) for f in FIELDS] + [sim.obs_log()["collisions"]]
    for a, b in zip(out["incremental"], out["full"]):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("n", [1000, 32767, 32768, 32769, 36865])
@pytest.mark.parametrize("dt,cut,lpc", [(1e-6, False, 1), (1e-6, True, 3), (1e-4, True, 1), (1e-4, False, 2)])
def test_fp64_steps_equal_calls(n, dt, cut, lpc):
    run = configs.Run(traps=[_trap(n, cut)], precision="fp64", energy_cut=cut, dt=dt, seed=3, lpc=lpc)
    if cut:
        run.traps[0].eta_end = run.traps[0].eta_start = 5.0   # constant: it does not matter when it is read
    with Simulation(run) as a, Simulation(run) as b:
        a.init_distribution()
        b.init_distribution()
        at = 0
        for steps in (1, 2 * lpc, 4 * lpc + 1, 3 * lpc):
            a.step(steps)
            for s in range(at, at + steps):
                if s % lpc == 0:
                    b.index_atoms()
                    b.sort_arrays()
                    b.build_cell_table()
                    b.collide()
                b.move_atoms()
                if cut:
                    b.evaporation_tag()
                    b.compact()
            at += steps
            for f in FIELDS + [_abi.FIELD_SIGVRMAX, _abi.FIELD_CELL_COUNT]:
                np.testing.assert_array_equal(a.copy_out(f), b.copy_out(f))
        a.step(2 * lpc)   # without a read in between
        a.step(5 * lpc)
