"""The pool of staging slabs (gh_slab_pool.h): small slabs do not keep large ones
out, a request takes the smallest that fits, devices are apart, the number kept is
bounded."""
from __future__ import annotations

import os
import subprocess

from conftest import ROOT

CSRC = os.path.join(ROOT, "gliomasolver_amd", "csrc")
PROGRAM = r"""
#include <cstdio>
#include "gh_slab_pool.h"
struct Slab { int id = 0, device = 0; size_t bytes = 0; };
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
    const size_t small = 128u << 10, large = 512u << 10;
    gh::SlabPool<Slab> pool;
    Slab s;
    CHECK(!pool.take(0, 1, s));
    for (int i = 0; i < 12; ++i) CHECK(pool.give({i, 0, small}) == (i < 8));  // many small transfers at once
    for (int i = 0; i < 12; ++i) CHECK(pool.give({100 + i, 0, large}) == (i < 8));
    CHECK(pool.ready(0, large) == 8 && pool.ready(0, small) == 8 && pool.slabs.size() == 16);
    CHECK(!pool.take(1, 1, s));
    CHECK(pool.give({200, 1, large}));
    for (int i = 0; i < 8; ++i) CHECK(pool.take(0, small, s) && s.bytes == small);
    CHECK(pool.ready(0, large) == 8);
    for (int i = 0; i < 4; ++i) CHECK(pool.take(0, small + 1, s) && s.bytes == large && s.device == 0);
    for (int i = 0; i < 4; ++i) CHECK(pool.take(0, 1, s) && s.bytes == large);  // no small one left
    CHECK(!pool.take(0, 1, s) && pool.slabs.size() == 1 && !pool.take(1, large + 1, s));
    return 0;
}
"""


def test_slab_pool(tmp_path):
    src, exe = tmp_path / "pool.cpp", tmp_path / "pool"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
