"""How many tokens a model's prefill buffers hold (memvanta_amd/host/step_plan.hpp): no more than its chunks where none
of them can join, within the stated bound on the scores, and a smaller step where memory is short, so that a model whose
single chunks fit still opens."""
import os
import subprocess

from conftest import ROOT

PROG = r"""
#include <cstdio>
#include <initializer_list>
#include "step_plan.hpp"
using namespace memvanta::hip;
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
    for (bool q8 : {false, true})
        for (std::size_t ctx : {1, 40, 256, 2048, 32768, 163840})
            for (std::size_t mb = 1; mb <= 600; ++mb) {
                const std::size_t s = step_tokens(mb, 256, ctx, 32, q8);
                bool any = false;  // some chunk size of this model joins
                for (std::size_t b = 1; b <= mb; ++b) any |= batch_joins(b, q8);
                CHECK(s >= mb && (any || s == mb));
                CHECK(s == mb || s <= 32 || s * 32 * ctx * 4 <= (std::size_t{512} << 20));
                if (any && mb < 256 && ctx == 2048) CHECK(s == 256);
                // with room for `room` tokens: a step that fits whenever the chunks do
                for (std::size_t room = mb > 3 ? mb - 3 : 1; room < 2 * mb + 300; room += 7) {
                    const std::size_t f = fit_step(s, mb, [&](std::size_t n) { return n <= room; });
                    CHECK(room >= mb ? f >= mb && f <= room && (f == s || 2 * f + 1 > room || f == mb) : f == 0);
                }
            }
    puts("ok");
    return 0;
}
"""


def test_step_tokens(tmp_path):
    src = tmp_path / "plan.cpp"
    src.write_text(PROG)
    exe = tmp_path / "plan"
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "memvanta_amd", "host"), "-o", str(exe),
                    str(src)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout
