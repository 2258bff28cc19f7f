"""Host side of the readbacks (csrc/kg_stage.h; no GPU needed).

A program compiled against the header checks which mappings a processor's copy
may go to."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "crystalgrowth_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "kg_stage.h"

static int bad = 0;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); bad = 1; } } while (0)

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

int main()
{
    pages();
    if (!bad)
        std::printf("ok\n");
    return bad;
}
"""


def test_pages(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "pages.cpp", tmp_path / "pages"
    src.write_text(PROGRAM)
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-g", "-Wall", "-Werror", "-I", CSRC,
                        str(src), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
