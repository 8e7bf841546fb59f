"""Work shared out to host threads (csrc/host_threads.hpp), compiled for the
host with allocations that fail: whichever one fails while the threads are
made, the work is done by those there are and the process goes on."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]
SRC = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include "host_threads.hpp"

static std::atomic<int> left{ 1 << 30 };   // allocations until one fails
void *operator new(std::size_t n)
{
    if (left.fetch_sub(1) == 0) throw std::bad_alloc();
    void *p = std::malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

int main()
{
    for (int threads = 1; threads <= 6; ++threads)
        for (int fail = 0; fail <= threads + 1; ++fail) {
            std::atomic<int> next{ 0 }, done{ 0 };
            auto work = [&](int) {
                while (next.fetch_add(1) < 100) done.fetch_add(1);
            };
            left = fail;
            dsmc::run_threads(threads, work);
            left = 1 << 30;
            if (done != 100) return 1;
        }
    std::puts("ok");
    return 0;
}
"""


def test_work_is_done_without_the_threads_that_cannot_be_made(tmp_path):
    (tmp_path / "t.cpp").write_text(SRC)
    exe = tmp_path / "t"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-pthread", f"-I{ROOT / 'cudadsmc_amd' / 'csrc'}",
                    str(tmp_path / "t.cpp"), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0 and res.stdout == "ok\n", (res.returncode, res.stderr)
