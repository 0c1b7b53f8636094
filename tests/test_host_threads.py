"""Parallel host sections (mts_threads.h) finish without memory: a thread that
cannot be started leaves its share to the others, and nothing is thrown (the C
functions that use them let no exception out)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include "mts_threads.h"
static std::atomic<int> left{-1};  // allocations until they fail (-1: never)
void* operator new(std::size_t n) {
    if (left >= 0 && left.fetch_sub(1) <= 0) {
        left = 0;
        throw std::bad_alloc();
    }
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
int main(int, char** argv) {
    const int nt = std::atoi(argv[1]);
    std::atomic<int> next{0}, done[100] = {};
    const int n = 100, a = 1, b = 2, c = 3;  // (captures larger than a small-function buffer)
    left = std::atoi(argv[2]);
    mts::on_threads(nt, [&, a, b, c](int) {
        for (int k; (k = next.fetch_add(1)) < n;) done[k] += a + b + c;
    });
    left = -1;
    for (int k = 0; k < n; k++)
        if (done[k] != 6) return 1;
    std::puts("ok");
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("threads")
    (d / "t.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-I" + os.path.join(ROOT, "mantiis_amd", "csrc"), str(d / "t.cpp"), "-o",
                    str(d / "t"), "-lpthread"], check=True, timeout=300)
    return str(d / "t")


@pytest.mark.parametrize("allocations", [-1, 0, 1, 2, 3, 5])
@pytest.mark.parametrize("threads", [1, 2, 8, 20])
def test_every_item_once_whatever_fails(exe, threads, allocations):
    r = subprocess.run([exe, str(threads), str(allocations)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stderr)
