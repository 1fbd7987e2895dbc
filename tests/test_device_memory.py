"""The blocks of device memory that a context keeps (ytrc_memory.h), on the
CPU: the header compiled against an allocator that counts what is held.

* With a budget, what the context holds, kept blocks included, stays within
  it, and what is refused depends only on what is in use, as without kept
  blocks.
* Without one, at most 96 MiB in 8 blocks of at most 32 MiB are kept.
* An allocation that finds no room on the device takes every context's kept
  blocks before it fails, also while other threads get and put blocks.
"""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r"""
#pragma once
#include <cstdint>
#include <cstdlib>
#include <map>
#include <mutex>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
inline std::map<void *, size_t> g_live;
inline uint64_t g_held = 0, g_size = UINT64_MAX;  // of the device
inline std::mutex g_mu;
inline hipError_t hipMalloc(void **p, size_t n)
{
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_held + n > g_size) return hipErrorOutOfMemory;
    *p = malloc(1);
    g_live[*p] = n;
    g_held += n;
    return hipSuccess;
}
inline hipError_t hipFree(void *p)
{
    std::lock_guard<std::mutex> lk(g_mu);
    auto it = g_live.find(p);
    if (it == g_live.end()) abort();
    g_held -= it->second;
    g_live.erase(it);
    free(p);
    return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
"""

BUDGET = r"""
#include <cstdio>
#include <random>
#include "ytrc_memory.h"
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
struct Block { char *p; size_t cap, bytes; };
int main()
{
    std::mt19937 rng(7);
    auto size = [&] { return (size_t)(rng() % 3 ? (1u << (rng() % 26)) : 1 + rng() % (40u << 20)); };
    for (uint64_t budget : {(uint64_t)0, (uint64_t)1 << 20, (uint64_t)50 << 20, (uint64_t)300 << 20}) {
        {
            DeviceMemory m;
            m.budget = budget;
            std::vector<Block> out;
            uint64_t used = 0, other = 0;  // of blocks, and of what is allocated elsewhere (masks, servers)
            for (int step = 0; step < 20000; step++) {
                const int what = (int)(rng() % 8);
                if (what < 3) {  // a pool, a batch
                    const size_t n = size();
                    CHECK(m.fits(n) == (budget == 0 || used + other + n <= budget));
                    if (!m.fits(n)) continue;
                    Block b{nullptr, 0, n};
                    CHECK(m.get(n, n, &b.p, &b.cap) == hipSuccess);
                    CHECK(g_live.count(b.p) && g_live[b.p] == b.cap && b.cap >= n);
                    CHECK(budget == 0 ? b.cap / 2 <= n : b.cap == n);
                    for (const Block &o : out) CHECK(o.p != b.p);
                    m.used += n;
                    used += n;
                    out.push_back(b);
                } else if (what < 6 && !out.empty()) {
                    const size_t k = rng() % out.size();
                    m.used -= out[k].bytes;
                    used -= out[k].bytes;
                    m.put(out[k].p, out[k].cap);
                    out.erase(out.begin() + (long)k);
                } else if (what == 6) {  // fields on their way into a dataset: beside the budget, for the call
                    const size_t n = size();
                    Block b{nullptr, 0, n};
                    CHECK(m.get(n, n, &b.p, &b.cap) == hipSuccess);
                    m.put(b.p, b.cap);
                } else if (rng() % 2) {  // a server
                    const size_t n = size();
                    if (!m.fits(n)) continue;
                    m.make_room(n);
                    m.used += n;
                    other += n;
                } else {
                    m.used -= other;
                    other = 0;
                }
                CHECK(m.used == used + other);
                uint64_t mine = 0;
                for (const Block &b : out) mine += b.cap;
                CHECK(budget == 0 || g_held + other <= budget);
                CHECK(g_held - mine <= DeviceMemory::KEPT_TOTAL);
                CHECK(g_live.size() - out.size() <= DeviceMemory::KEPT_COUNT);
            }
            for (const Block &b : out) m.put(b.p, b.cap);
        }
        CHECK(g_held == 0 && g_live.empty());
    }
    puts("ok");
    return 0;
}
"""

FULL = r"""
#include <cstdio>
#include <thread>
#include "ytrc_memory.h"
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main()
{
    const size_t MB = 1u << 20;
    g_size = 100 * MB;
    {
        DeviceMemory a, b;
        struct { char *p; size_t cap; } keep[3];
        for (int i = 0; i < 3; i++) CHECK((i ? a : b).get(30 * MB, 30 * MB, &keep[i].p, &keep[i].cap) == hipSuccess);
        for (int i = 0; i < 3; i++) (i ? a : b).put(keep[i].p, keep[i].cap);
        CHECK(g_held == 90 * MB);
        // a server's arena, a mask: neither is a kept block
        float *arena = nullptr;
        CHECK(DeviceMemory::alloc(&arena, 95 * MB) == hipSuccess);
        CHECK(g_held == 95 * MB);
        char *p;
        size_t cap;
        CHECK(a.get(6 * MB, 6 * MB, &p, &cap) == hipErrorOutOfMemory);
        CHECK(b.get(5 * MB, 5 * MB, &p, &cap) == hipSuccess);
        b.put(p, cap);
        hipFree(arena);
        // (one context's blocks for another's)
        CHECK(a.get(98 * MB, 98 * MB, &p, &cap) == hipSuccess);
        a.put(p, cap);
    }
    CHECK(g_held == 0);
    std::vector<std::thread> threads;
    std::atomic<int> bad{0};
    for (int t = 0; t < 6; t++)
        threads.emplace_back([&, t] {
            DeviceMemory m;
            for (int i = 0; i < 3000; i++) {
                char *p;
                size_t cp;
                // (a block is at most twice as large as asked for: at most
                // 6 (8 + 4) of 100 MB are out at once)
                const size_t n = (size_t)(1 + (i * 7 + t) % 4) * MB;
                if (m.get(n, n, &p, &cp) != hipSuccess) bad++;
                else {
                    float *r;
                    if (DeviceMemory::alloc(&r, 4 * MB) != hipSuccess) bad++;
                    else hipFree((char *)r);
                    m.put(p, cp);
                }
            }
        });
    for (auto &t : threads) t.join();
    CHECK(g_held == 0 && g_live.empty());
    puts("ok");
    return 0;
}
"""


def _run(tmp_path, source):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(source)
    exe = str(tmp_path / "main")
    subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", "-I", str(tmp_path), "-I", os.path.join(ROOT, "yt_amd", "csrc"),
                    str(tmp_path / "main.cpp"), "-o", exe], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr
    assert res.stdout == "ok\n"


def test_kept_blocks_stay_within_the_budget(tmp_path):
    _run(tmp_path, BUDGET)


def test_no_allocation_fails_for_kept_blocks(tmp_path):
    _run(tmp_path, FULL)
