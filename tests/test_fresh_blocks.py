"""The lists of allocations that are made ahead (csrc/fresh_blocks.hpp) against a pool that runs out, refuses and fails to wait, on
the CPU."""
import pathlib
import subprocess

CSRC = pathlib.Path(__file__).parents[1] / "ai-ml-emulation-layer-for-vulkan_amd" / "csrc"
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <set>
#include "fresh_blocks.hpp"
using mlel::FreshBlocks;
enum Error { ok, no_memory, captured, lost };
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); std::exit(1); } } while (0)
struct Pool {
    FreshBlocks blocks;
    std::set<void *> live, uncleared;
    int left = 1 << 30, waits = 0;
    Error refusal = ok, wait_result = ok;
    Error take(void **out) {
        *out = nullptr;
        return blocks.take(out, no_memory,
            [&](void **p) {
                if (refusal != ok) return refusal;
                if (left == 0) return no_memory;
                left--, *p = std::malloc(16), live.insert(*p), uncleared.insert(*p);
                return ok;
            },
            [&] { waits++; if (wait_result == ok) uncleared.clear(); return wait_result; },
            [&](void *p) { drop(p); });
    }
    void drop(void *p) { CHECK(live.erase(p) == 1); uncleared.erase(p); std::free(p); left++; }
    void *good() {
        void *p;
        CHECK(take(&p) == ok && p != nullptr && live.count(p) && !uncleared.count(p));
        CHECK(given.insert(p).second);
        return p;
    }
    std::set<void *> given;
    ~Pool() {
        for (void *p : given) drop(p);
        blocks.clear([&](void *p) { drop(p); });
        CHECK(live.empty());
    }
};
int main() {
    {   // apart, cleared, and as many to a wait as are made ahead
        Pool pool;
        for (int i = 0; i < 100; i++) pool.good();
        CHECK(pool.waits == (100 + mlel::kFreshBlocks - 1) / mlel::kFreshBlocks);
    }
    for (int before = 0; before <= 17; before++) {  // refused whatever lies ready, and taken again
        Pool pool;
        void *p;
        for (int i = 0; i < before; i++) pool.good();
        pool.refusal = captured;
        for (int i = 0; i < 3; i++) CHECK(pool.take(&p) == captured && p == nullptr);
        pool.refusal = ok;
        for (int i = 0; i < 20; i++) pool.good();
    }
    for (int memory = 0; memory <= 40; memory++) {  // whatever was made is handed out before there is none
        Pool pool;
        void *p;
        pool.left = memory;
        for (int i = 0; i < memory; i++) pool.good();
        CHECK(pool.take(&p) == no_memory && p == nullptr);
        pool.left = 3;
        for (int i = 0; i < 3; i++) pool.good();
        CHECK(pool.take(&p) == no_memory && p == nullptr);
    }
    for (int before = 0; before <= 17; before++) {  // a wait that fails hands nothing out and keeps nothing
        Pool pool;
        void *p;
        for (int i = 0; i < before; i++) pool.good();
        pool.wait_result = lost;
        Error e = ok;
        for (int i = 0; i < 9 && e == ok; i++) { e = pool.take(&p); if (e == ok) pool.given.insert(p); }
        CHECK(e == lost && p == nullptr && pool.uncleared.empty() && pool.live.size() == pool.given.size());
        pool.wait_result = ok;
        for (int i = 0; i < 20; i++) pool.good();
    }
    std::puts("done");
}
"""


def test_lists(tmp_path):
    source, program = tmp_path / "lists.cpp", tmp_path / "lists"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(source), "-o", str(program)], check=True)
    out = subprocess.run([str(program)], capture_output=True, text=True)
    assert out.stdout.strip() == "done", out.stdout + out.stderr
