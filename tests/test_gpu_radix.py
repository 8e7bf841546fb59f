"""The primitives where their plans change: digits of 8 or 10 bits, tiles of
2048 or 4096 pairs, the ends of tiles; and calls on several threads and
streams at once, which must not share scratch."""
import ctypes as C
import threading

import numpy as np
import pytest

from cudadsmc_amd import load_library
from gpu_util import DeviceArray

pytestmark = pytest.mark.gpu


def _sort(lib, k, v, bits, stream=None):
    with DeviceArray(lib, k) as dk, DeviceArray(lib, v) as dv:
        assert lib.dsmc_sort_by_key(dk.ptr, dv.ptr, len(k), bits, stream) == 0
        return dk.get(), dv.get()


@pytest.mark.parametrize("n", [1, 2047, 2049, 4096, 4097, (1 << 18) - 1, 1 << 18, (1 << 18) + 1, 3 << 19, (3 << 19) + 1])
@pytest.mark.parametrize("bits", [8, 10, 17, 20, 21, 26, 32])
def test_sort_plans(n, bits):
    lib = load_library()
    rng = np.random.default_rng(n + bits)
    k = rng.integers(0, 1 << bits, n, dtype=np.uint64).astype(np.uint32)
    k[::3] = k[0]   # many equal keys: the order of their values shows stability
    v = np.arange(n, dtype=np.uint32)
    gk, gv = _sort(lib, k, v, bits)
    order = np.argsort(k, kind="stable")
    np.testing.assert_array_equal(gk, k[order])
    np.testing.assert_array_equal(gv, order.astype(np.uint32))


@pytest.mark.parametrize("n", [1, 2047, 2048, 2049, 8193, 1 << 20])
@pytest.mark.parametrize("p", [0.0, 0.3, 1.0])
def test_remove_if_and_scan_tiles(n, p):
    lib = load_library()
    rng = np.random.default_rng(n)
    v = rng.integers(-9, 9, n).astype(np.int32)
    st = (rng.random(n) < p).astype(np.int32) * 7
    m = C.c_int(-1)
    with DeviceArray(lib, v) as dv, DeviceArray(lib, st) as ds, DeviceArray(lib, np.zeros(n, np.int32)) as do:
        assert lib.dsmc_exclusive_scan(dv.ptr, do.ptr, n, None) == 0
        np.testing.assert_array_equal(do.get(), np.concatenate([[0], np.cumsum(v)[:-1]]).astype(np.int32))
        assert lib.dsmc_remove_if(dv.ptr, ds.ptr, n, C.byref(m), None) == 0
        assert m.value == int((st == 0).sum())
        np.testing.assert_array_equal(dv.get()[:m.value], v[st == 0])


def test_calls_on_threads_do_not_share_scratch():
    lib = load_library()
    hip = C.CDLL("libamdhip64.so.7")   # the runtime that the library has loaded
    bad = []

    def work(seed):
        rng = np.random.default_rng(seed)
        stream = C.c_void_p()
        assert hip.hipStreamCreate(C.byref(stream)) == 0
        for r in range(12):
            n = int(rng.integers(1, 300000))
            k = rng.integers(0, 1 << 20, n).astype(np.uint32)
            v = np.arange(n, dtype=np.uint32)
            # copies on the default stream end before the sort's stream starts
            gk, gv = _sort(lib, k, v, 20, stream)
            order = np.argsort(k, kind="stable")
            if not (np.array_equal(gk, k[order]) and np.array_equal(gv, order)):
                bad.append((seed, r, n))
        done.append(hip.hipStreamDestroy(stream))

    done = []
    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad and done == [0, 0, 0, 0]
