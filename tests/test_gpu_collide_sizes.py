"""The collide's slots per lane (two, four or eight by the context's capacity)
and its block size (by the number of traps) on both sides of each limit.  FP32:
a trap's run does not depend on the traps beside it, so a trap alone in a small
context (two slots per lane) is compared, bitwise, with the same trap in
contexts whose other traps take them over each limit; FP64: the whole step
against the same loop call by call."""
import numpy as np
import pytest

from cudadsmc_amd import Simulation, _abi, configs

pytestmark = pytest.mark.gpu

FIELDS = [_abi.FIELD_POS, _abi.FIELD_VEL, _abi.FIELD_ATOM_ID, _abi.FIELD_SIGVRMAX]


def _box(precision, n, nc):
    box = configs.box_thermalise(precision, n, nc).traps[0]
    box.n_real = 2.5e12   # n sigma <v_r> dt = 0.2 collisions per atom and step
    return box


def _first_trap(n, nc, others):
    """State of the first trap (n atoms) after three steps, and its collisions."""
    base = configs.box_thermalise("fp32", n, nc)
    run = base.with_(traps=[_box("fp32", n, nc)] + [_box("fp32", m, 3) for m in others], dt=2e-6)
    rng = np.random.default_rng(n)   # the first trap's atoms first: the same in every context
    parts = [(rng.uniform(-1.0, 1.0, (m, 3)), rng.normal(0.0, 0.05, (m, 3))) for m in (n, sum(others))]
    pos = np.concatenate([p for p, _ in parts]) * np.array(run.traps[0].half_width)
    vel = np.concatenate([v for _, v in parts])
    with Simulation(run) as sim:
        sim.set_state(pos, vel)
        sim.step(3)
        out = [sim.copy_out(f)[:n] for f in FIELDS[:3]] + [sim.copy_out(FIELDS[3])[:nc ** 3]]
        return out + [sim.obs_log()["collisions"][:, 0].copy()]


@pytest.mark.parametrize("others", [[(1 << 17) - 5000], [1 << 17], [3 << 17], [300] * 519, [760] * 519])
@pytest.mark.parametrize("n", [2, 127, 129, 513, 5000])
def test_fp32_trap_beside_others(n, others):
    print(f"fp32 n={n} others={others[0]} x {len(others)}", flush=True)
    for nc in (1, 3, 9):
        alone = _first_trap(n, nc, [])
        beside = _first_trap(n, nc, others)
        if n > 500:
            assert alone[4].sum() > n // 100
        for a, b in zip(alone, beside):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("n", [1 << 17, (1 << 17) + 1, 3 << 17, (3 << 17) + 1])
def test_fp32_one_large_trap(n):
    print(f"fp32 n={n}", flush=True)
    alone, beside = _first_trap(n, 20, []), _first_trap(n, 20, [2])
    assert alone[4].sum() > n // 100
    for a, b in zip(alone, beside):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("n", [127, 129, 1 << 19, (1 << 19) + 1, (1 << 19) + 513])
def test_fp64_slots_per_lane(n):
    print(f"fp64 n={n}", flush=True)
    run = configs.box_thermalise("fp64", n, 20 if n > 1000 else 3).with_(dt=2e-6)
    run.traps[0].n_real = 2.5e12
    with Simulation(run) as a, Simulation(run) as b:
        a.init_distribution()
        b.init_distribution()
        a.step(3)
        for _ in range(3):
            b.index_atoms()
            b.sort_arrays()
            b.build_cell_table()
            b.collide()
            b.move_atoms()
        if n > 1000:
            assert a.obs_log()["collisions"].sum() > n // 100
        for f in FIELDS + [_abi.FIELD_COLLISION_COUNT]:
            np.testing.assert_array_equal(a.copy_out(f), b.copy_out(f))
