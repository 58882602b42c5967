"""The pool of idle pinned blocks (csrc/nb_idle_pool.h), compiled for the host:
the bound counts each device's own blocks, and the pool empties with its last
holder."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "astronbodysim.jl_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include <set>
#include "nb_idle_pool.h"
struct B { int dev; B *next; };
#define CHECK(c) do { if (!(c)) { std::printf("%s\n", #c); return 1; } } while (0)
int main() {
    static nb::IdlePool<B, 4> pool;
    static B b[8][5];
    for (int d = 0; d < 8; ++d)
        for (int k = 0; k < 5; ++k) b[d][k].dev = d;
    CHECK(!pool.give(&b[0][0]));                     // nobody holds the pool
    pool.hold();
    pool.hold();
    for (int round = 0; round < 3; ++round) {
        for (int d = 0; d < 8; ++d)
            for (int k = 0; k < 5; ++k) CHECK(pool.give(&b[d][k]) == (k < 4));
        for (int d = 7; d >= 0; --d) {
            std::set<B *> got;
            for (int k = 0; k < 4; ++k) {
                B *p = pool.take(d);
                CHECK(p && p->dev == d);
                got.insert(p);
            }
            CHECK(got.size() == 4 && !pool.take(d));
        }
    }
    CHECK(pool.give(&b[2][0]) && pool.give(&b[6][1]));
    CHECK(!pool.release());
    B *p = pool.release();
    CHECK(p && p->next && !p->next->next && p->dev + p->next->dev == 8);
    CHECK(!pool.take(2) && !pool.give(&b[2][0]));
    return 0;
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="needs g++")
def test_idle_blocks_per_device(tmp_path):
    (tmp_path / "pool.cpp").write_text(PROGRAM)
    exe = tmp_path / "pool"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-pthread", f"-I{CSRC}", str(tmp_path / "pool.cpp"),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
