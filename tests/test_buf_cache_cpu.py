"""The cache of idle buffers, compiled for the host with a counting allocator:
a buffer stays with the device it was allocated on, is reused by requests it
holds with at most twice their size, and the cap bounds what is kept."""
import subprocess

from conftest import ROOT

PROGRAM = r"""
#include <assert.h>
#include <stdio.h>
#include <stdlib.h>
#include "buf_cache.hpp"

static int device = 0, live = 0;
struct Memory {
    void* alloc(size_t bytes) { ++live; return malloc(16 + bytes * 0); }
    void free(void* p) { --live; ::free(p); }
    int place() { return device; }
};

int main() {
    const size_t mb = size_t(1) << 20;
    zg::BufCache<Memory> cache(64 * mb);
    size_t got = 0;
    void* a = cache.acquire(8 * mb, &got);
    assert(a && got == 8 * mb && live == 1);
    cache.release(a, got);
    // another device current: not the first one's buffer
    device = 1;
    void* b = cache.acquire(8 * mb, &got);
    assert(b && b != a && live == 2);
    cache.release(b, got);
    // each device gets its own back, whatever order they were released in
    device = 0;
    void* c = cache.acquire(7 * mb, &got);
    assert(c == a && got == 8 * mb);
    device = 1;
    void* d = cache.acquire(7 * mb, &got);
    assert(d == b && got == 8 * mb && live == 2);
    cache.release(d, got);
    device = 0;
    cache.release(c, got);
    // too large for the request: a new one
    void* e = cache.acquire(1 * mb, &got);
    assert(e != a && got == 2 * mb && live == 3);
    cache.release(e, got);
    // past the cap: given back at once
    void* f = cache.acquire(60 * mb, &got);
    assert(live == 4);
    cache.release(f, got);
    assert(live == 3);
    cache.free_all();
    assert(live == 0);
    puts("ok");
}
"""


def test_buffers_stay_on_their_device(tmp_path):
    src, exe = tmp_path / "cache.cpp", tmp_path / "cache"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", str(ROOT / "zynum_amd" / "csrc"), str(src), "-o", str(exe)],
                   check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout == "ok\n"
