"""What a context keeps of its calls' memory, with counted allocations in place
of the device's: a small program of the header that holds the rules."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bayadera_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "bh_pool.hpp"

struct Memory {
    static inline size_t used = 0, limit = (size_t)1 << 40, allocs = 0;
    static int alloc(void** p, size_t n, bool) {
        if (used + n > limit) return 2;
        used += n;
        ++allocs;
        size_t* h = (size_t*)std::malloc(sizeof(size_t));
        *h = n;
        *p = h;
        return 0;
    }
    static void release(void* p, bool) {
        used -= *(size_t*)p;
        std::free(p);
    }
};
using Pool = bh::Pool<Memory>;
constexpr size_t MiB = (size_t)1 << 20;

// one call that holds `n` blocks of these sizes at once; 0 or the error
int call(Pool& pool, const size_t* bytes, int n, bool pinned = false) {
    Pool::Block b[8];
    int rc = 0, held = 0;
    for (; held < n && rc == 0; ++held) rc = pool.get(bytes[held], pinned, &b[held]);
    if (rc) --held;
    for (int i = 0; i < held; ++i) pool.put(b[i]);
    return rc;
}
size_t allocs_of(Pool& pool, const size_t* bytes, int n, int times) {
    const size_t before = Memory::allocs;
    for (int i = 0; i < times; ++i) call(pool, bytes, n);
    return Memory::allocs - before;
}

int main() {
    const size_t small[3] = {16, 200000, 1 * MiB}, large[2] = {40 * MiB, 5000}, draws[1] = {64 * MiB};
    {   // small calls after one that staged 40 MB: their blocks are kept
        Pool pool;
        call(pool, large, 2);
        allocs_of(pool, small, 3, 1);
        std::printf("after_large %zu\n", allocs_of(pool, small, 3, 10));
        // and the large one's are, beside them
        allocs_of(pool, draws, 1, 1);
        std::printf("large_beside %zu\n", allocs_of(pool, draws, 1, 10) + allocs_of(pool, small, 3, 10));
    }
    {   // more sizes than are kept, then other ones
        Pool pool;
        for (int e = 0; e < 9; ++e) {
            size_t s[8];
            for (size_t& v : s) v = (size_t)4096 << e;
            call(pool, s, 8);
        }
        const size_t other[1] = {3 * MiB};
        allocs_of(pool, other, 1, 1);
        std::printf("stale_sizes %zu\n", allocs_of(pool, other, 1, 10));
    }
    {   // bounded, whatever comes
        Pool pool;
        size_t most = 0;
        for (int i = 0; i < 300; ++i) {
            const size_t s[3] = {(size_t)(i * 977 % 90 + 1) * MiB, (size_t)i * 5003 + 1, MiB};
            call(pool, s, 3);
            call(pool, s + 1, 1, true);
            if (Memory::used > most) most = Memory::used;
        }
        std::printf("bounded %d\n", most <= Pool::kDevMax + Pool::kPinMax && pool.kept.size() <= Pool::kBlocks);
    }
    {   // what is kept does not make a call fail that would fit without it
        Memory::limit = 100 * MiB;
        Pool pool, other;
        call(other, draws, 1);
        const size_t need[2] = {20 * MiB, 90 * MiB};
        call(pool, need, 1);
        std::printf("short_of_memory %d\n", call(pool, need + 1, 1));
        const size_t never[1] = {101 * MiB};
        std::printf("refused %d\n", call(pool, never, 1) != 0);
        Memory::limit = (size_t)1 << 40;
    }
    {   // what is only of use goes first: where it is not held, and not for its like
        Memory::limit = 100 * MiB;
        Pool pool;
        const size_t need[1] = {90 * MiB};
        bh::Extra<Memory> a, b;
        a.take({30 * MiB, 10 * MiB});
        b.take({50 * MiB, 20 * MiB});  // the second of them does not fit
        std::printf("extra_taken %d\n", a.there() && !b.there() && Memory::used == 40 * MiB);
        {
            auto held = a.hold();
            std::printf("extra_held %d\n", call(pool, need, 1) != 0 && a.there());
        }
        std::printf("extra_given %d\n", call(pool, need, 1) == 0 && !a.there());
        Memory::limit = (size_t)1 << 40;
    }
    std::printf("left %zu\n", Memory::used);
    return 0;
}
"""


@pytest.fixture(scope="module")
def result(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    (d / "pool.cpp").write_text(PROGRAM)
    cxx = shutil.which("g++") or "/opt/rocm/bin/amdclang++"
    subprocess.run([cxx, "-std=c++17", "-O1", "-I", CSRC, str(d / "pool.cpp"), "-o", str(d / "pool"), "-lpthread"],
                   check=True)
    out = subprocess.run([str(d / "pool")], check=True, capture_output=True, text=True, timeout=60).stdout
    return dict(line.split() for line in out.splitlines())


@pytest.mark.parametrize("what,value", [
    ("after_large", 0), ("large_beside", 0), ("stale_sizes", 0), ("bounded", 1), ("short_of_memory", 0),
    ("refused", 1), ("extra_taken", 1), ("extra_held", 1), ("extra_given", 1), ("left", 0)])
def test_kept_blocks(result, what, value):
    assert int(result[what]) == value
