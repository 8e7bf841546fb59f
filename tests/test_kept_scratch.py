"""Device memory that the primitives keep idle between calls goes back before
an allocation of the library fails.  Runs without a GPU: in a process of its
own the HIP calls that a primitive makes are taken by a stand-in that counts
allocated bytes up to a limit and launches nothing."""
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]
HIP = r"""
#include <stddef.h>
#include <stdint.h>
typedef struct { uint32_t x, y, z; } dim3_t;
static size_t used, size[64];
static const size_t limit = (size_t)1 << 30;
int hipMalloc(void **p, size_t n)
{
    for (int i = 0; i < 64; ++i)
        if (!size[i]) {
            if (used + n > limit) return 2;
            used += size[i] = n;
            *p = (void *)((uintptr_t)(i + 1) << 40);
            return 0;
        }
    return 2;
}
int hipFree(void *p)
{
    const int i = (int)((uintptr_t)p >> 40) - 1;
    used -= size[i];
    size[i] = 0;
    return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned f) { static int64_t mem[8]; *p = mem; return 0; }
int hipHostFree(void *p) { return 0; }
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipGetLastError(void) { return 0; }
int hipStreamSynchronize(void *s) { return 0; }
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t l, void *s) { return 0; }
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *l, void **s)
{
    g->x = g->y = g->z = b->x = b->y = b->z = 1;
    *l = 0;
    *s = 0;
    return 0;
}
int hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **a, size_t l, void *s) { return 0; }
size_t bytes_used(void) { return used; }
"""
CHECK = r"""
import ctypes as C, sys
hip = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
hip.bytes_used.restype = C.c_size_t
lib = C.CDLL(sys.argv[2])
lib.dsmc_device_alloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
lib.dsmc_device_free.argtypes = [C.c_void_p]
lib.dsmc_sort_by_key.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_void_p]
keys = C.c_void_p(1 << 50)
assert lib.dsmc_sort_by_key(keys, keys, 30000000, 24, None) == 0
kept = hip.bytes_used()
assert 200 << 20 < kept <= 512 << 20, kept
p = C.c_void_p()
assert lib.dsmc_device_alloc(C.byref(p), (1 << 30) - (100 << 20)) == 0
assert hip.bytes_used() == (1 << 30) - (100 << 20)
q = C.c_void_p()
assert lib.dsmc_device_alloc(C.byref(q), 200 << 20) == 3      # DSMC_ENOMEM
assert lib.dsmc_device_free(p) == 0
assert lib.dsmc_device_alloc(C.byref(q), 200 << 20) == 0
assert lib.dsmc_device_free(q) == 0 and hip.bytes_used() == 0
"""


def test_device_alloc_takes_the_kept_scratch_back(tmp_path):
    (tmp_path / "hip.c").write_text(HIP)
    so = tmp_path / "libhip_standin.so"
    subprocess.run(["gcc", "-O1", "-fPIC", "-shared", "-w", str(tmp_path / "hip.c"), "-o", str(so)], check=True)
    res = subprocess.run([sys.executable, "-c", CHECK, str(so), str(ROOT / "cudadsmc_amd" / "libdsmc.so")],
                         capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stderr
