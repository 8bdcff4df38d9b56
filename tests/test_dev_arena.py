"""A roadmap's device memory (dev_arena.hpp) against a stand-in for hipMalloc:
every range lies inside one live block and meets no other, whatever the order
of sizes and whichever requests the device refuses.  No GPU calls."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HARNESS = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>

#include "dev_arena.hpp"

// addresses only: a block's memory is never touched
static std::map<char *, size_t> live;
static char *next_address = (char *)0x100000;
static int refuse_from = -1, refuse_count = 0, calls = 0;

extern "C" hipError_t hipMalloc(void **p, size_t n)
{
    const int k = calls++;
    if (k >= refuse_from && k < refuse_from + refuse_count)
        return hipErrorOutOfMemory;
    *p = next_address;
    live[next_address] = n;
    next_address += n + 4096 - n % 4096 + 4096; // blocks never touch
    return hipSuccess;
}
extern "C" hipError_t hipFree(void *p)
{
    if (!live.erase((char *)p)) {
        std::printf("freed what is not held\n");
        std::exit(1);
    }
    return hipSuccess;
}
extern "C" hipError_t hipGetLastError() { return hipSuccess; }

static std::map<char *, size_t> held;

static void check(void *v, size_t n, const char *what)
{
    char *p = (char *)v;
    auto b = live.upper_bound(p);
    const bool in = b != live.begin() && (--b, p + n <= b->first + b->second);
    auto above = held.lower_bound(p);
    bool apart = above == held.end() || p + n <= above->first;
    if (above != held.begin()) {
        auto below = above;
        --below;
        apart = apart && below->first + below->second <= p;
    }
    if (!in || !apart) {
        std::printf("%s: %zu bytes %s\n", what, n, in ? "meet another range" : "leave their block");
        std::exit(1);
    }
    held[p] = n;
}

static void run(const char *what, const std::vector<size_t> &sizes, int from = -1, int count = 0)
{
    refuse_from = from;
    refuse_count = count;
    calls = 0;
    held.clear();
    {
        pump::rmb::DevArena a;
        // before the requests, room for the first three, which one block then holds
        if (sizes.size() > 3)
            a.reserve({sizes[2], sizes[0], sizes[1]});
        const size_t before = live.size();
        std::vector<std::pair<void *, size_t>> got;
        int served = 0;
        for (size_t n : sizes) {
            void *p = a.alloc(n);
            if (!p) {
                if (!count) {
                    std::printf("%s: refused without cause\n", what);
                    std::exit(1);
                }
                continue;
            }
            check(p, n, what);
            got.push_back({p, n});
            if (!count && sizes.size() > 3 && ++served == 3 && live.size() != before) {
                std::printf("%s: reserved room not used\n", what);
                std::exit(1);
            }
            if (got.size() % 3 == 0) { // every third request gives the first one back
                a.release(got[0].first);
                held.erase((char *)got[0].first);
                got.erase(got.begin());
                if (void *w = a.alloc_whole(n)) { // goes back at once, whatever its size
                    const size_t with = live.size();
                    check(w, n, what);
                    a.release(w);
                    held.erase((char *)w);
                    if (live.size() + 1 != with) {
                        std::printf("%s: not given back\n", what);
                        std::exit(1);
                    }
                }
            }
        }
    }
    if (!live.empty()) {
        std::printf("%s: blocks left behind\n", what);
        std::exit(1);
    }
}

int main()
{
    const size_t M = (size_t)1 << 20;
    run("first past the first block", {12 * M, 15 * M, 100, 9 * M, 16 * M, 16 * M + 1, 1});
    run("first block full", {8 * M, 1, 8 * M, 8 * M, 8 * M, 8 * M + 1, 32 * M, 256});
    run("just past", {8 * M + 1, 8 * M - 255, 255, 257});
    for (int from = 0; from < 5; ++from)
        for (int count = 1; count < 4; ++count)
            run("refused", {12 * M, 12 * M, 100, 20 * M, 12 * M, 15 * M, 9 * M, 64 * M, 3}, from, count);
    std::mt19937 g(1);
    for (int r = 0; r < 300; ++r) {
        std::vector<size_t> s;
        for (int k = 0; k < 60; ++k) // up to 31 MiB, spread over the logarithm
            s.push_back(1 + g() % ((size_t)1 << (1 + g() % 25)));
        run("random", s, r % 2 ? (int)(g() % 8) : -1, r % 2 ? (int)(g() % 3) : 0);
    }
    std::printf("ok\n");
    return 0;
}
"""


def test_ranges_lie_in_their_blocks(tmp_path):
    src, exe = tmp_path / "arena.cpp", tmp_path / "arena"
    src.write_text(HARNESS)
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "pump_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
