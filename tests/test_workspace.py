"""The growth of the library's stream workspaces (brain_amd/csrc/bh_ws_grow.h),
compiled alone with an allocator that counts and can run out: what slowly rising
sizes leave behind stays below twice the buffer in use, and a failed growth leaves the
buffer as it was."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "brain_amd", "csrc")

MAIN = r"""
#include "bh_ws_grow.h"
#include <cstdio>
#include <cstdlib>
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)
int main() {
    static int mem[1];
    size_t total = 0, calls = 0, limit = SIZE_MAX;
    auto alloc = [&](size_t bytes) -> void* {
        ++calls;
        if (bytes > limit) return nullptr;
        total += bytes / 4;
        return mem;
    };
    const size_t cap = 100000;
    bh::WsBuf b;
    for (size_t n = 333; n <= cap; ++n) {  // every size in turn
        CHECK(bh::ws_grow(b, n, cap, alloc));
        CHECK(b.ints >= n && b.ints <= cap && b.ws == mem);
        CHECK(total - b.ints < 2 * b.ints);  // left behind
    }
    CHECK(calls < 12 && b.ints == cap);
    CHECK(bh::ws_grow(b, cap + 1, cap, alloc) && b.ints == cap + 1);  // one call may need more
    // No memory for twice the size, then for none.
    bh::WsBuf c;
    CHECK(bh::ws_grow(c, 1000, cap, alloc) && c.ints == 1000);
    limit = 1200 * 4;
    CHECK(bh::ws_grow(c, 1100, cap, alloc) && c.ints == 1100);
    limit = 0;
    CHECK(!bh::ws_grow(c, 1300, cap, alloc) && c.ints == 1100 && c.ws == mem);
    CHECK(bh::ws_grow(c, 1100, cap, alloc));
    return 0;
}
"""


def test_workspace_growth(tmp_path):
    src, exe = tmp_path / "ws.cpp", tmp_path / "ws"
    src.write_text("#include <cstdint>\n" + MAIN)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
