"""The pool of pinned host memory that solvers and batches share
(alsvinn_amd/csrc/avh_pinned.hpp), with an allocator that keeps count, on the
CPU: slots are distinct and used again, more of them than a page holds come as
allocations of their own, several threads take and give them, and the page goes
with the last holder, whether that is the context or a solver."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>
#include <thread>
#include <vector>
#include "avh_pinned.hpp"
using namespace avh;
static std::mutex m;
static std::set<void*> live;
static int bad = 0;
static void* take(size_t n) { std::lock_guard<std::mutex> g(m); void* p = malloc(n); live.insert(p); return p; }
static void drop(void* p) {
    std::lock_guard<std::mutex> g(m);
    if (!live.erase(p)) { ++bad; printf("released what was not allocated\n"); return; }
    memset(p, 0xee, PINNED_SLOT);
    free(p);
}
static void* none(size_t) { return nullptr; }
#define CHECK(x) do { if (!(x)) { ++bad; printf("line %d: %s\n", __LINE__, #x); } } while (0)
int main() {
    {   // the context's handle goes first; a solver writes through its slot afterwards
        auto ctx = std::make_shared<PinnedPool>(take, drop);
        auto* solver = new PinnedSlot;
        auto* batch = new PinnedSlot;
        char* p = (char*)solver->take(ctx);
        char* q = (char*)batch->take(ctx);
        CHECK(p && q && p != q);
        ctx.reset();
        CHECK(live.size() == 1);
        memset(p, 1, PINNED_SLOT);
        delete solver;
        CHECK(live.size() == 1);
        memset(q, 2, PINNED_SLOT);
        delete batch;
        CHECK(live.empty());
    }
    {   // the solver goes first; its slot is taken again
        auto ctx = std::make_shared<PinnedPool>(take, drop);
        void* p;
        { PinnedSlot s; p = s.take(ctx); }
        { PinnedSlot s; CHECK(s.take(ctx) == p); }
        CHECK(live.size() == 1);
        ctx.reset();
        CHECK(live.empty());
    }
    {   // more than a page holds
        auto ctx = std::make_shared<PinnedPool>(take, drop);
        std::vector<PinnedSlot> s(PINNED_SLOTS + 3);
        std::set<void*> at;
        for (auto& x : s) at.insert(x.take(ctx));
        CHECK(at.size() == s.size() && live.size() == 4);
        ctx.reset();
        for (void* a : at) memset(a, 3, PINNED_SLOT);
        s = std::vector<PinnedSlot>();
        CHECK(live.empty());
    }
    {   // threads
        auto ctx = std::make_shared<PinnedPool>(take, drop);
        std::vector<std::thread> t;
        for (int k = 0; k < 8; ++k)
            t.emplace_back([&ctx, k] {
                for (int i = 0; i < 2000; ++i) {
                    PinnedSlot a, b;
                    char* p = (char*)a.take(ctx);
                    char* q = (char*)b.take(ctx);
                    memset(p, k, PINNED_SLOT);
                    memset(q, k + 8, PINNED_SLOT);
                    for (size_t c = 0; c < PINNED_SLOT; ++c)
                        if (p[c] != k || q[c] != k + 8) { std::lock_guard<std::mutex> g(m); ++bad; }
                }
            });
        for (auto& x : t) x.join();
        ctx.reset();
        CHECK(live.empty());
    }
    {   // no memory
        auto ctx = std::make_shared<PinnedPool>(none, drop);
        PinnedSlot s;
        CHECK(!s.take(ctx));
    }
    return bad ? 1 : 0;
}
"""


def test_pool_outlives_whoever_goes_first(tmp_path):
    src = tmp_path / "pool.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "pool"
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-pthread", "-I",
                    os.path.join(ROOT, "alsvinn_amd", "csrc"), "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
