"""Threads of one C call (the read-back of the model): with no memory or no thread to be had for one, its share is done by
the caller, every thread has ended and no exception leaves (CPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <atomic>
#include <cstdlib>
#include <new>
#include <system_error>
#include "host/shared_work.h"
static std::atomic<int> left{-1};  // allocations until one fails (-1: never)
static bool system_err = false;
void *operator new(std::size_t n)
{
    if (left >= 0 && left-- == 0) {
        if (system_err) throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
        throw std::bad_alloc();
    }
    return std::malloc(n);
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }
extern "C" int run(int threads)
{
    int done[4] = {0, 0, 0, 0};
    emc::run_shared<4>(threads, [&](int t) { ++done[t]; });
    for (int t = 0; t < 4; ++t)
        if (done[t] != (t < threads ? 1 : 0)) return 1;
    return 0;
}
int main()
{
    int bad = run(1) + run(4);
    for (int err = 0; err < 2; ++err)
        for (int at = 0; at < 4; ++at) {
            system_err = err != 0;
            left = at;
            bad += run(4);
            left = -1;
        }
    return bad;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")
def test_shares_are_done_whatever_fails(tmp_path):
    src, exe = tmp_path / "shared.cpp", tmp_path / "shared"
    src.write_text(SRC)
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "emc_amd", "csrc"), str(src), "-o", str(exe),
                        "-lpthread"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stderr[-2000:])
