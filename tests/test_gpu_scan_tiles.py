"""Scan, removal and compaction map on both sides of the number of tiles
(12288 of 2048) up to which every block adds up the tiles before its own and
above which their sums are scanned first; and the time, which must not grow
with the square of the tiles."""
import ctypes as C
import time

import numpy as np
import pytest

from cudadsmc_amd import Simulation, _abi, configs, load_library
from gpu_util import DeviceArray

pytestmark = pytest.mark.gpu

LIMIT = 12288 * 2048


@pytest.mark.parametrize("n", [LIMIT - 1, LIMIT, LIMIT + 1, LIMIT + 2048, LIMIT + 2049, 2 * LIMIT + 12345])
@pytest.mark.parametrize("p", [0.0, 0.3, 1.0])
def test_scan_and_removal(n, p):
    lib = load_library()
    rng = np.random.default_rng(n)
    v = rng.integers(-9, 9, n, dtype=np.int32)
    st = (rng.random(n, dtype=np.float32) < p).astype(np.int32) * 7
    expect = np.zeros(n, np.int32)
    np.cumsum(v[:-1], dtype=np.int32, out=expect[1:])
    m = C.c_int(-1)
    with DeviceArray(lib, v) as dv, DeviceArray(lib, st) as ds, DeviceArray(lib, v) as do:
        assert lib.dsmc_exclusive_scan(do.ptr, do.ptr, n, None) == 0   # in place
        assert np.array_equal(do.get(), expect)
        assert lib.dsmc_remove_if(dv.ptr, ds.ptr, n, C.byref(m), None) == 0
        assert m.value == int((st == 0).sum())
        assert np.array_equal(dv.get()[:m.value], v[st == 0])


@pytest.mark.parametrize("n", [LIMIT, LIMIT + 1])
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_reads_of_a_run_with_losses(n, precision):
    """A read drops the removed atoms through the compaction map: every label
    is either among those read or has the record of a removed atom."""
    trap = configs.quadrupole_trap(n, 64, n_real=1e9)
    trap.eta_start = trap.eta_end = 5.0
    trap.T_cut = trap.T
    with Simulation(configs.Run(traps=[trap], precision=precision, energy_cut=True, dt=1e-6, seed=2)) as sim:
        sim.init_distribution()
        sim.step(2)
        ids, key = sim.copy_out(_abi.FIELD_ATOM_ID), sim.copy_out(_abi.FIELD_CELL_ID)
        alive = sim.info().n_alive
        lost = np.flatnonzero(sim.copy_out(_abi.FIELD_EVAP_POS).any(axis=1))
    assert 0 < alive < n and len(ids) == len(key) == alive and len(lost) == n - alive
    held = np.zeros(n, np.int8)
    held[ids] += 1
    held[lost] += 1
    assert held.min() == held.max() == 1
    assert key.max() < trap.nc[0] * trap.nc[1] * trap.nc[2] + 1


def test_time_grows_with_the_elements():
    """Four times the elements, about four times the time (nearly nine times
    when every block adds up the earlier tiles)."""
    lib = load_library()
    best = {}
    with DeviceArray(lib, np.zeros(0, np.int32)) as a, DeviceArray(lib, np.zeros(0, np.int32)) as b:
        for d in (a, b):
            lib.dsmc_device_free(d.ptr)
            assert lib.dsmc_device_alloc(C.byref(d.ptr), 4 << 30) == 0
        for n in (1 << 28, 1 << 30):
            for _ in range(4):
                t = time.perf_counter()
                assert lib.dsmc_exclusive_scan(a.ptr, b.ptr, n, None) == 0
                best[n] = min(best.get(n, 1e9), time.perf_counter() - t)
    print({n: f"{t * 1e3:.2f} ms" for n, t in best.items()}, flush=True)
    assert best[1 << 30] < 6.0 * best[1 << 28]
