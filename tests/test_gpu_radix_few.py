"""The radix sort around the number of tiles (32 of 2048 or 4096 pairs) up to
which a pass has no scan launch of its own: numpy's stable argsort, with one
and several passes of both digit widths and with many equal keys."""
import numpy as np
import pytest

from tests.gpu_util import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2047, 2049, 65535, 65536, 65537, 131071, 131072, 131073])
@pytest.mark.parametrize("bits", [1, 8, 16, 20, 31])
def test_sorts_by_key(lib, n, bits):
    rng = np.random.default_rng(n + bits)
    keys = rng.integers(0, 1 << bits, size=n, dtype=np.uint64).astype(np.uint32)
    vals = rng.permutation(n).astype(np.uint32)
    with DeviceArray(lib, keys) as dk, DeviceArray(lib, vals) as dv:
        assert lib.dsmc_sort_by_key(dk.ptr, dv.ptr, n, bits, None) == 0
        order = np.argsort(keys, kind="stable")
        np.testing.assert_array_equal(dk.get(), keys[order])
        np.testing.assert_array_equal(dv.get(), vals[order])
