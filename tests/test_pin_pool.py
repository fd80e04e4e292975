"""The pool of pinned blocks behind the one-token calls with host vectors (memvanta_amd/host/pin_pool.hpp), with a
counting allocator on the host: one block for any number of objects that call in turn, more only while calls overlap,
a bound on what lies free, and no block out twice."""
import os
import subprocess

from conftest import ROOT

PROG = r"""
#include <atomic>
#include <cstdio>
#include <set>
#include <thread>
#include "pin_pool.hpp"
static std::atomic<int> made{0}, live{0};
static bool full = false;
struct A {
    static uint8_t* make() {
        if (full) return nullptr;
        ++made, ++live;
        return new uint8_t[8]{};
    }
    static void drop(uint8_t* p) { --live; delete[] p; }
};
using Pool = memvanta::hip::PinPool<A>;
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
    {
        Pool p(3);
        for (int object = 0; object < 100; ++object) {  // each one's first call
            uint8_t* b = p.take();
            CHECK(b && p.give(b));
        }
        CHECK(made == 1);
        uint8_t* b[5];
        for (auto& q : b) q = p.take();
        CHECK(made == 5 && (std::set<uint8_t*>(b, b + 5).size()) == 5);
        CHECK(p.give(b[0]) && p.give(b[1]) && p.give(b[2]) && !p.give(b[3]) && !p.give(b[4]));
        A::drop(b[3]), A::drop(b[4]);
        p.trim(1);
        CHECK(live == 1);
        CHECK(p.take() && live == 1);
        full = true;
        CHECK(!p.take());
        full = false;
    }
    Pool p(8);
    made = 0;
    std::atomic<int> clash{0};
    std::thread t[6];
    for (int i = 0; i < 6; ++i)
        t[i] = std::thread([&, i] {
            for (int k = 0; k < 20000; ++k) {
                uint8_t* b = p.take();
                b[0] = static_cast<uint8_t>(i + 1);
                b[1] = static_cast<uint8_t>(k);
                if (b[0] != i + 1 || b[1] != static_cast<uint8_t>(k)) ++clash;
                b[0] = 0;
                if (!p.give(b)) ++clash;
            }
        });
    for (auto& x : t) x.join();
    CHECK(clash == 0 && made <= 6);
    puts("ok");
    return 0;
}
"""


def test_blocks_are_shared_and_bounded(tmp_path):
    src = tmp_path / "pool.cpp"
    src.write_text(PROG)
    exe = tmp_path / "pool"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "memvanta_amd", "host"), "-o",
                    str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout
