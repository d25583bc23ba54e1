"""The cutting of device reads into launches and slots (cellsim3d_amd/csrc/cs3d_read.h)
on the CPU: every word of every segment goes to its place once, pieces lie aligned and
apart inside their slots, no launch holds more pieces than it can; and where the host's
memory runs out at any of its allocations, it says so instead of throwing."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
static long g_left = -1;  // allocations until memory runs out (-1: never)
void* operator new(size_t n) {
    if (g_left == 0) throw std::bad_alloc();
    if (g_left > 0) --g_left;
    void* p = std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void* operator new[](size_t n) { return operator new(n); }
void operator delete(void* p) noexcept { std::free(p); }
void operator delete[](void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }
void operator delete[](void* p, size_t) noexcept { std::free(p); }
#include "cs3d_read.h"
using namespace cs3d;
static unsigned rnd(unsigned& s) { return s = s * 1664525u + 1013904223u, s >> 8; }
int main() {
    unsigned seed = 7;
    long cases = 0, bad = 0, refused = 0, finished = 0;
    const size_t slot = 4096;
    for (int it = 0; it < 2000; ++it) {
        const int n = 1 + rnd(seed) % 30;
        std::vector<std::vector<uint32_t>> dev(n), host(n);
        std::vector<ReadSeg> segs;
        size_t total = 0;
        for (int i = 0; i < n; ++i) {
            const size_t edge[8] = {0, 1, 4, 1023, 1024, 1025, 1020, 2048};
            const size_t w = rnd(seed) % 3 ? edge[rnd(seed) % 8] : rnd(seed) % 5000;
            dev[i].resize(w);
            for (auto& v : dev[i]) v = rnd(seed);
            host[i].assign(w, 0);
            segs.push_back(ReadSeg{dev[i].data(), host[i].data(), 4 * w});
            total += 4 * w;
        }
        ReadPlan p;
        bad += !plan_reads(segs.data(), n, slot, p) || p.total != total || p.lists.size() != p.pieces.size();
        std::vector<char> buf(slot), used(slot);
        for (size_t k = 0; k < p.lists.size(); ++k) {  // as k_gather and the host copy
            const GatherList& g = p.lists[k];
            bad += g.n < 1 || g.n > kMaxGather || (size_t)g.n != p.pieces[k].size() || p.done[k].load() != 0;
            std::fill(used.begin(), used.end(), 0);
            for (int j = 0; j < g.n; ++j) {
                const size_t at = 4 * (size_t)g.dst[j], len = 4 * (size_t)g.words[j];
                if (at % 16 || at + len > slot) { ++bad; continue; }
                for (size_t b = at; b < at + len; ++b) bad += used[b]++;
                std::memcpy(buf.data() + at, g.src[j], len);
            }
            for (const ReadPiece& q : p.pieces[k]) std::memcpy(q.host, buf.data() + q.off, q.bytes);
        }
        for (int i = 0; i < n; ++i) bad += dev[i] != host[i];
        ++cases;
        if (it % 20) continue;
        for (long left = 0;; ++left) {
            ReadPlan q;
            g_left = left;
            const bool ok = plan_reads(segs.data(), n, slot, q);
            g_left = -1;
            if (ok) { ++finished; break; }
            ++refused;
        }
    }
    std::printf("%ld %ld %ld %ld\n", cases, bad, refused, finished);
    return 0;
}
"""


def test_read_plans_place_every_word_and_survive_short_memory(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    src = tmp_path / "plan_check.cpp"
    src.write_text(SRC)
    exe = tmp_path / "plan_check"
    subprocess.run([cxx, "-std=c++17", "-O1", "-I", os.path.join(ROOT, "cellsim3d_amd", "csrc"), "-o",
                    str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=300).stdout
    print(out)
    cases, bad, refused, finished = (int(v) for v in out.split())
    assert (cases, bad, finished) == (2000, 0, 100) and refused > 300
