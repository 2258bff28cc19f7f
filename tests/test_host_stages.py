"""Host side of the readbacks (csrc/kg_stage.h; no GPU needed).

A program compiled against the header checks which mappings a processor's copy
may go to, and that the pool of buffers gives each to one call at a time, frees
what it allocated, and lets other calls pass while one waits for its memory."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "crystalgrowth_amd", "csrc")

PROGRAM = r"""
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <future>
#include <thread>
#include <vector>
#include "kg_stage.h"

static int bad = 0;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); bad = 1; } } while (0)

static std::atomic<int> allocated{0}, waiting{0};
static std::atomic<bool> open_{true};
static void *get(size_t n)
{
    if (n == kg::StagePool::STAGE_MAX) {
        ++waiting;
        while (!open_)
            std::this_thread::yield();
    }
    ++allocated;
    return std::malloc(n);
}
static void put(void *p)
{
    --allocated;
    std::free(p);
}

static void pages()
{
    const size_t n = (size_t)sysconf(_SC_PAGESIZE);
    auto map = [&](int prot) {
        return static_cast<char *>(mmap(nullptr, 4 * n, prot, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
    };
    char *rw = map(PROT_READ | PROT_WRITE), *ro = map(PROT_READ), *none = map(PROT_NONE);
    // (a kernel without the call says so of every mapping)
    const bool known = madvise(rw, n, MADV_POPULATE_WRITE) == 0;
    CHECK(kg::populate(rw, 4 * n) == known);
    CHECK(kg::populate(rw + 13, 2 * n) == known);
    CHECK(!kg::populate(ro, 4 * n));
    CHECK(!kg::populate(ro + 5, 1));
    CHECK(!kg::populate(none, 4 * n));
    mprotect(rw + 2 * n, n, PROT_READ);   // one page in the middle
    CHECK(!kg::populate(rw, 4 * n));
    CHECK(kg::populate(rw, 2 * n) == known);
    munmap(none, 4 * n);
    CHECK(!kg::populate(none, 4 * n));
}

static void others_pass_while_one_waits()
{
    kg::StagePool pool(get, put);
    pool.retain();
    const int first = pool.take(400 << 10);
    CHECK(first == 0 && pool.capacity(first) == (size_t)1 << 20);
    pool.give(first);
    open_ = false;
    std::thread large([&] {
        const int at = pool.take(3 << 20);
        CHECK(at >= 0 && pool.capacity(at) == kg::StagePool::STAGE_MAX);
        pool.give(at);
    });
    while (waiting == 0)
        std::this_thread::yield();
    // the buffer that grows is not given to anyone; a small copy gets its own
    std::future<int> small = std::async(std::launch::async, [&] { return pool.take(400 << 10); });
    const bool passed = small.wait_for(std::chrono::seconds(20)) == std::future_status::ready;
    CHECK(passed);
    open_ = true;
    large.join();
    CHECK(small.get() != first);
    pool.release();
    CHECK(allocated == 0);
}

static void one_call_at_a_time()
{
    kg::StagePool pool(get, put);
    pool.retain();
    std::atomic<int> taken{0};
    std::vector<std::thread> t;
    for (int k = 0; k < 12; ++k)
        t.emplace_back([&, k] {
            for (int i = 0; i < 2000; ++i) {
                const size_t n = (size_t)1 << (10 + (k + i) % 13);
                const int at = pool.take(n);
                if (at < 0)
                    continue;
                ++taken;
                const size_t m = n < pool.capacity(at) ? n : pool.capacity(at);
                std::memset(pool.buffer(at), k, m);
                std::this_thread::yield();
                for (size_t q = 0; q < m; q += 509)
                    CHECK(pool.buffer(at)[q] == (char)k);
                pool.give(at);
            }
        });
    for (auto &q : t)
        q.join();
    CHECK(taken > 0 && allocated <= kg::StagePool::STAGES);
    pool.release();
    CHECK(allocated == 0);
}

static void no_memory()
{
    kg::StagePool pool([](size_t) -> void * { return nullptr; }, put);
    pool.retain();
    CHECK(pool.take(1 << 20) == -1);
    CHECK(pool.take(1 << 20) == -1);   // and the slot is free again
    pool.release();
}

int main()
{
    pages();
    others_pass_while_one_waits();
    one_call_at_a_time();
    no_memory();
    if (!bad)
        std::printf("ok\n");
    return bad;
}
"""


def test_pages_and_buffers(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "stages.cpp", tmp_path / "stages"
    src.write_text(PROGRAM)
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-g", "-Wall", "-Werror", "-pthread", "-I", CSRC,
                        str(src), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
