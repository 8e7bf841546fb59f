"""Host reads on both sides of the size from which several threads copy them
(16 MB), and whole and partial last pieces (2 MB): equal to a read into pinned
memory, which is copied directly, also while another context is read by
another thread."""
import ctypes as C
import threading

import numpy as np
import pytest

from cudadsmc_amd import Simulation, _abi, configs

pytestmark = pytest.mark.gpu

# rows of 24 bytes: just below 16 MB, at it, one row over, whole pieces, and more
SIZES = [(16 << 20) // 24, (16 << 20) // 24 + 1, (18 << 20) // 24, (18 << 20) // 24 + 1, 2000003]


class Pinned:
    """n rows of three doubles in memory pinned by the library's own runtime."""

    def __init__(self, n):
        self.hip = C.CDLL("libamdhip64.so.7")
        self.ptr = C.c_void_p()
        assert self.hip.hipHostMalloc(C.byref(self.ptr), C.c_size_t(24 * n), C.c_uint(0)) == 0
        self.rows = np.ctypeslib.as_array(C.cast(self.ptr, C.POINTER(C.c_double)), (n, 3))

    def close(self):
        self.rows = None
        assert self.hip.hipHostFree(self.ptr) == 0


def _read(sim, field, out):
    _abi.check(sim.lib, sim.lib.dsmc_copy_out(sim.h, field, out.ctypes.data_as(C.c_void_p), out.nbytes), sim.h)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("n", SIZES)
def test_large_reads(n, precision):
    print(f"large reads n={n} {precision}", flush=True)
    rng = np.random.default_rng(n)
    pos, vel = rng.normal(0.0, 1e-4, (n, 3)), rng.normal(0.0, 0.05, (n, 3))
    run = configs.Run(traps=[configs.quadrupole_trap(n, 20)], precision=precision)
    with Simulation(run) as a, Simulation(run) as b:
        a.set_state(pos, vel)
        b.set_state(vel, pos)
        got = [np.full((n, 3), np.nan) for _ in range(4)]
        other = threading.Thread(target=lambda: [_read(b, f, o) for f, o in
                                                 ((_abi.FIELD_POS, got[2]), (_abi.FIELD_VEL, got[3]))])
        other.start()
        _read(a, _abi.FIELD_POS, got[0])
        _read(a, _abi.FIELD_VEL, got[1])
        other.join()
        pinned = Pinned(n)
        for sim, field, g in ((a, _abi.FIELD_POS, got[0]), (a, _abi.FIELD_VEL, got[1]),
                              (b, _abi.FIELD_POS, got[2]), (b, _abi.FIELD_VEL, got[3])):
            pinned.rows[:] = np.nan
            _read(sim, field, pinned.rows)
            np.testing.assert_array_equal(g, pinned.rows)
        pinned.close()
