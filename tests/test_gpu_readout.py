"""Host reads and writes of the state at the edges of tiles and blocks: the
rows of dsmc_copy_out against the same numbers laid out with numpy, with every
atom alive and with removed atoms still in their slots."""
import numpy as np
import pytest

from cudadsmc_amd import Simulation, _abi, configs

pytestmark = pytest.mark.gpu

SIZES = [1, 63, 64, 65, 255, 257, 2047, 2049]


def _atoms(n, seed=3):
    rng = np.random.default_rng(seed)
    return rng.normal(0, 2e-5, (n, 3)), rng.normal(0, 0.04, (n, 3))


def _split(v):
    hi = v.astype(np.float32)
    return hi, (v - hi.astype(np.float64)).astype(np.float32)


def _round13(r):
    """Round to nearest-even with the low 11 mantissa bits clear."""
    u = r.view(np.uint32).astype(np.uint64)
    return (((u + 0x3FF + ((u >> 11) & 1)) & 0xFFFFF800).astype(np.uint32)).view(np.float32)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("form", ["fp64", "fp32"])
def test_rows_of_given_atoms(form, n):
    pos, vel = _atoms(n)
    run = configs.Run(traps=[configs.quadrupole_trap(n, 9)], precision=form, spin=True)
    with Simulation(run) as sim:
        sim.set_state(pos, vel)
        spin = np.random.default_rng(5).normal(size=(n, 3 if form == "fp32" else 4))
        sim.set_spin(spin)
        got = [sim.copy_out(f) for f in (_abi.FIELD_POS, _abi.FIELD_VEL, _abi.FIELD_ATOM_ID, _abi.FIELD_SPIN)]
        sv = sim.copy_out(_abi.FIELD_SIGVRMAX)
        if form == "fp32":
            rem = sim.copy_out(_abi.FIELD_POS_COMP), sim.copy_out(_abi.FIELD_VEL_COMP)
    if form == "fp32":
        (ph, pl), (vh, vl) = _split(pos), _split(vel)
        pl = _round13(pl)
        pos, vel = ph.astype(float) + pl, vh.astype(float) + vl
        spin = spin.astype(np.float32).astype(float)
        np.testing.assert_array_equal(rem[0], pl.astype(float))
        np.testing.assert_array_equal(rem[1], vl.astype(float))
    for a, b in zip(got, (pos, vel, np.arange(n), spin)):
        np.testing.assert_array_equal(a, b)
    t = run.traps[0]
    s0 = np.sqrt(16. * configs.KB * t.T / (configs.PI_REF * run.mass)) * run.sigma
    s0 = float(np.float32(s0)) if form == "fp32" else s0
    np.testing.assert_allclose(sv[:9 ** 3 + 1], s0, rtol=0 if form == "fp32" else 1e-15)
    assert sv[9 ** 3 + 1] == 0.0


@pytest.mark.parametrize("n", SIZES)
def test_rows_beside_removed_atoms(n):
    """One FP32 step with a cut between the atoms' energies: the reads skip the
    removed slots, keep the slot order and agree with each other."""
    pos, vel = _atoms(n)
    trap = configs.quadrupole_trap(n, 9)
    e = 0.5 * configs.MRB * (vel ** 2).sum(1) + trap.mu * trap.dBdz * np.sqrt(
        pos[:, 0] ** 2 + pos[:, 1] ** 2 + 4 * pos[:, 2] ** 2)
    trap.T_cut, trap.eta_start = trap.T, float(np.median(e)) / (configs.KB * trap.T) * (1 + 1e-3)
    trap.eta_end = trap.eta_start
    run = configs.Run(traps=[trap], precision="fp32", energy_cut=True, sigma=0.0, dt=1e-9)
    keep = e <= trap.eta_start * configs.KB * trap.T
    with Simulation(run) as sim:
        sim.set_state(pos, vel)
        sim.step(1)
        ids, p, c = (sim.copy_out(f) for f in (_abi.FIELD_ATOM_ID, _abi.FIELD_POS, _abi.FIELD_CELL_ID))
        start = sim.copy_out(_abi.FIELD_TRAP_START)
        assert sim.info().n_alive == keep.sum()
        # unsorted moves leave no trap table behind: the count is then taken
        # from the keys
        sim.index_atoms()
        assert sim.info().n_alive == keep.sum()
        np.testing.assert_array_equal(sim.copy_out(_abi.FIELD_ATOM_ID), ids)
    np.testing.assert_array_equal(np.sort(ids), np.flatnonzero(keep))
    np.testing.assert_allclose(p, pos[ids], rtol=0, atol=1e-9)
    assert (np.diff(c) >= 0).all()      # dt moves no atom to another cell
    np.testing.assert_array_equal(start, [0, keep.sum()])
