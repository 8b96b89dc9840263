"""The pool of staging slots (csrc/sp_slots.h), built for the CPU with memory
that counts and can be made to fail: a later call allocates nothing, a failed
request leaves no slot behind, what exceeds the bound is freed, and no slot is
lent to two threads at once."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "stochastic-parker_amd", "csrc")

PROGRAM = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>
#include "sp_slots.h"

std::atomic<int> allocs{0}, live{0}, left{1 << 30};
struct Mem {
    static int get(void** p, size_t bytes) {
        if (left.fetch_sub(1) <= 0) return 2;
        *p = std::malloc(bytes);
        ++allocs; ++live;
        return 0;
    }
    static void drop(void* p) { std::free(p); --live; }
};
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)

int main() {
    sp::SlotPool<Mem, 8> pool;
    void* a[16];
    CHECK(pool.take(a, 8) == 0 && allocs == 8);
    pool.give(a, 8);
    CHECK(pool.take(a, 5) == 0 && allocs == 8);      // a later call allocates nothing
    pool.give(a, 5);
    left = 2;                                        // eight idle slots and two more
    CHECK(pool.take(a, 11) == 2 && live == 8);       // the slots it had are back, the surplus freed
    left = 1 << 30;
    const int before = allocs;
    CHECK(pool.take(a, 8) == 0 && allocs == before);
    void* b[16];
    CHECK(pool.take(b, 16) == 0 && live == 24);
    pool.give(a, 8);
    pool.give(b, 16);
    CHECK(live == 8);                                // bounded
    std::atomic<int> shared{0};
    std::vector<std::thread> ts;
    for (int t = 0; t < 8; ++t)
        ts.emplace_back([&, t] {
            void* s[5];
            for (int i = 0; i < 4000; ++i) {
                const int n = 1 + (i + t) % 5;
                if (pool.take(s, n) != 0) { ++shared; continue; }
                for (int k = 0; k < n; ++k) *static_cast<volatile int*>(s[k]) = 100 * t + k;
                std::this_thread::yield();
                for (int k = 0; k < n; ++k)
                    if (*static_cast<volatile int*>(s[k]) != 100 * t + k) ++shared;
                pool.give(s, n);
            }
        });
    for (auto& t : ts) t.join();
    CHECK(shared == 0 && live <= 8);
    std::puts("ok");
    return 0;
}
"""

def test_slot_pool(tmp_path):
    src, exe = tmp_path / "pool.cpp", tmp_path / "pool"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-pthread",
                    "-I", CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout
