"""The policy of held flow memory (csrc/flow_blocks.h) with a device of a few
megabytes in place of the runtime: compiled and run on the CPU."""
import os
import subprocess

from conftest import ROOT

PROGRAM = r"""
#include <cassert>
#include <cstdio>
#include <map>

#include "flow_blocks.h"

static size_t room = 64u << 20;
static std::map<void*, size_t> live;

struct Device {
    static void* alloc(size_t bytes) {
        if (bytes > room) return nullptr;
        static size_t next = 0;  // never the same address again
        void* p = reinterpret_cast<void*>(next += 64);
        live[p] = bytes;
        room -= bytes;
        return p;
    }
    static void release(void* p) {
        auto it = live.find(p);
        assert(it != live.end());  // once, and only its own
        room += it->second;
        live.erase(it);
    }
};
using Blocks = nbx::FlowBlocks<Device>;

int main() {
    constexpr size_t MB = 1u << 20;
    Blocks b;
    // a closed flow's block serves the next of its size or an eighth less
    b.open();
    b.open();
    auto a = b.take(9 * MB);
    b.close({a, {nullptr, 0}}, true);
    assert(room == 55 * MB);
    b.open();
    auto c = b.take(8 * MB);
    assert(c.p == a.p && c.bytes == 9 * MB);
    b.close({c}, true);
    b.open();
    auto d = b.take(7 * MB);  // too small for it
    assert(d.p != a.p && room == 48 * MB);
    // an allocation that fails gives back what is held and is tried again
    auto e = b.take(50 * MB);
    assert(e.p != nullptr && live.count(a.p) == 0 && room == 7 * MB);
    auto f = b.take(8 * MB);
    assert(f.p == nullptr && room == 7 * MB);
    b.close({d, f}, true);
    assert(room == 7 * MB);
    b.give_back();
    assert(room == 14 * MB && live.size() == 1);
    // nothing is held while its work may still run
    b.open();
    d = b.take(4 * MB);
    b.close({d}, false);
    assert(room == 14 * MB);
    // the last flow to close gives everything back
    b.open();
    d = b.take(4 * MB);
    b.close({d}, true);
    assert(room == 10 * MB);
    b.close({e}, true);
    assert(room == 64 * MB && live.empty());
    // at most kMostBytes are held
    room = 64 * Blocks::kMostBytes;
    b.open();
    b.open();
    d = b.take(Blocks::kMostBytes / 2);
    e = b.take(Blocks::kMostBytes / 2 + 1);
    b.close({d, e}, true);
    assert(room == 64 * Blocks::kMostBytes - Blocks::kMostBytes / 2 && live.size() == 1);
    b.close({}, true);
    assert(room == 64 * Blocks::kMostBytes);
    std::puts("ok");
    return 0;
}
"""


def test_flow_blocks(tmp_path):
    src, exe = tmp_path / "blocks.cc", tmp_path / "blocks"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-UNDEBUG",
                    "-I", os.path.join(ROOT, "numbacs_amd", "csrc"), "-o", str(exe), str(src)],
                   check=True)
    assert subprocess.run([str(exe)], check=True, capture_output=True).stdout == b"ok\n"
