"""The FP32 spin substeps where their fast and their guarded loop meet.

A wave whose atoms all stay off the field's zero and below the sine's
reduction range runs the substeps without tests; one with any other atom runs
them with the tests.  So an atom's spin must not depend, to the bit, on its
wave holding such an atom; and that atom itself must keep its spin at the
field's zero, or turn by its large angle.  Substep counts around the unrolled
loop's remainder, waves full and partial, with and without interpolation.

Tolerance at the large angle (no interpolation, so one axis and `substeps`
equal turns by phi): each FP32 angle carries a few roundings, phi 2^-24 each;
8 of them per turn, and as much again for the axis: substeps (phi + 4) 2^-20.
"""
import numpy as np
import pytest

from cudadsmc_amd import Simulation, _abi, configs

pytestmark = pytest.mark.gpu

HBAR, MUB = 1.05457148e-34, 9.27400915e-24


def turned(run, pos, vel, spin):
    with Simulation(run) as sim:
        sim.set_state(pos, vel)
        sim.set_spin(spin)
        sim.step(1)
        s = sim.copy_out(_abi.FIELD_SPIN)
        order = np.argsort(sim.copy_out(_abi.FIELD_ATOM_ID))
    return s[order]


@pytest.mark.parametrize("interp", [False, True])
@pytest.mark.parametrize("substeps", [1, 2, 3, 20])
@pytest.mark.parametrize("n", [2, 64, 300])
def test_guarded_wave_gives_the_same_spins(n, substeps, interp):
    run = configs.spin_evaporation("fp32", n_atoms=n, nc=4).with_(
        sigma=0.0, spin_loss=False, energy_cut=False, spin_substeps=substeps, spin_interp=interp,
        obs_capacity=8)
    tr = run.traps[0]
    rng = np.random.default_rng(100 * n + substeps)
    pos = rng.normal(0.0, 0.2, (n, 3)) * np.array(tr.half_width)
    vel = rng.normal(0.0, 0.05, (n, 3))
    spin = rng.normal(size=(n, 3))
    spin /= np.linalg.norm(spin, axis=1)[:, None]
    spin = spin.astype(np.float32).astype(np.float64)
    print(f"spin substeps n={n} substeps={substeps} interp={interp}", flush=True)
    plain = turned(run, pos, vel, spin)
    w = run.gs * MUB * (run.dt / substeps) / HBAR
    k = n // 2
    others = np.arange(n) != k

    # at the field's zero, at rest: the spin stays
    p, v = pos.copy(), vel.copy()
    p[k] = 0.0
    v[k] = 0.0
    zero = turned(run, p, v, spin)
    assert np.array_equal(zero[others], plain[others])
    assert np.max(np.abs(zero[k] - spin[k])) <= 2.0 ** -22   # (normalised again)

    # an angle beyond the reduction range
    phi = 9000.0
    p, v = pos.copy(), vel.copy()
    p[k] = 0.0
    p[k, 0] = np.float32(phi / (w * tr.dBdz))
    v[k] = 0.0
    far = turned(run, p, v, spin)
    assert np.array_equal(far[others], plain[others])
    if not interp:
        total = substeps * w * tr.dBdz * p[k, 0]
        c, s = np.cos(total), np.sin(total)
        e = np.array([1.0, 0.0, 0.0])
        want = spin[k] * c + np.cross(e, spin[k]) * s + e * spin[k, 0] * (1.0 - c)
        assert np.max(np.abs(far[k] - want)) <= substeps * (phi + 4.0) * 2.0 ** -20
