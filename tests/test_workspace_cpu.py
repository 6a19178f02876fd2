"""Growth of an executor's device buffers (csrc/workspace.h) with a stand-in for
device memory that refuses: a failed optional buffer is attempted once and
leaves everything as it was, and is given back for one that is needed."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cassert>
#include <cstdio>
#include <cstdlib>
#include <map>
#include "workspace.h"
using namespace srq;

struct Mem {  // `room` bytes in all
    size_t room, used = 0;
    int allocs = 0, syncs = 0;
    bool oom = false, lost = false;
    std::map<void *, size_t> live;
    bool alloc(void **p, size_t n) {
        ++allocs;
        if (used + n > room) return oom = true, false;
        *p = std::malloc(1);
        live[*p] = n, used += n;
        return true;
    }
    bool release(void *p) {
        assert(live.count(p));
        used -= live[p], live.erase(p), std::free(p);
        return true;
    }
    bool sync() { return ++syncs, !lost; }
    bool out_of_memory() const { return oom; }
};

int main() {
    {  // a needed buffer: at least 256 bytes, then by halves
        Mem m{1000000};
        DevBuf b;
        assert(grow(b, 10, m) && b.n == 256 && m.syncs == 0);
        assert(grow(b, 200, m) && m.allocs == 1);
        assert(grow(b, 300, m) && b.n == 384 && m.syncs == 1 && m.used == 384);
        assert(grow(b, 4000, m) && b.n == 4000);
    }
    {  // an optional one: exact, the old kept until the new is there
        Mem m{1000};
        OptionalBuf o;
        assert(grow_optional(o, 300, m) && o.n == 300);
        assert(grow_optional(o, 400, m) && o.n == 400 && m.used == 400 && m.syncs == 1);
        void *held = o.p;
        const int tried = m.allocs;
        assert(!grow_optional(o, 700, m) && m.allocs == tried + 1);
        assert(o.p == held && o.n == 400 && m.used == 400 && m.syncs == 1);  // no wait, nothing freed
        for (int i = 0; i < 5; ++i) assert(!grow_optional(o, 700 + i, m));
        assert(m.allocs == tried + 1);          // attempted once
        assert(grow_optional(o, 350, m));       // what it holds still serves
        assert(grow_optional(o, 550, m) && o.n == 550);  // less than was refused
    }
    {  // a device that stopped answering: the old stays, the new is not leaked
        Mem m{1000};
        OptionalBuf o;
        assert(grow_optional(o, 300, m));
        void *held = o.p;
        m.lost = true;
        assert(!grow_optional(o, 400, m) && o.p == held && o.n == 300 && m.used == 300);
    }
    {  // memory runs short for a needed buffer: the optional one makes way, and stays away
        Mem m{1000};
        DevBuf b;
        OptionalBuf o;
        assert(grow(b, 300, m) && grow_optional(o, 500, m));
        assert(grow_or_give_back(b, 600, o, m) && b.n == 600 && !o.p && o.n == 0);
        const int tried = m.allocs;
        assert(!grow_optional(o, 500, m) && m.allocs == tried);
        assert(grow_optional(o, 300, m));
        assert(!grow_or_give_back(b, 5000, o, m) && !o.p);  // not enough even so
    }
    {  // nothing to give back
        Mem m{100};
        DevBuf b;
        OptionalBuf o;
        assert(!grow_or_give_back(b, 500, o, m) && !b.p && b.n == 0 && m.allocs == 1);
    }
    std::puts("workspace ok");
}
"""


def test_growth_with_refused_allocations(tmp_path):
    (tmp_path / "t.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "t")
    r = subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "sr_go_tranformer_amd", "csrc"),
                        str(tmp_path / "t.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "workspace ok" in r.stdout, r.stderr
