"""The start steps of the fused path's spike lists (csrc/mgb_lists.h) in a CPU model of
persistent launches whose workgroups start late: each segment's workgroups wait only for
their own segment, so one segment may have ended its launch before another's first
workgroup has read the words that the launch before left."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MODEL = r"""
#include <cstdio>
#include <algorithm>
#include <numeric>
#include <vector>
#include "mgb_lists.h"
// A run of launches (windows, steps of each), segments in a fixed order: a workgroup of the
// segment's first tile writes each window's start, one of its last tile reads in the launch's
// first window, up to `ahead` windows later (one is what the segment's own wait allows).
// Every read has to give the window's start less the window before it.  SHARED: every
// segment uses segment 0's words.
static int run(int nseg, const std::vector<std::pair<int, int>>& launches, std::vector<int> order, int ahead) {
    std::vector<int64_t> tb(3 * nseg, 0);
    int64_t base = 0, window = 0, before = 0;   // first step and index of the launch, steps of the window before
    int wrong = 0;
    for (auto [nwin, nst] : launches) {
        for (int q : order) {
#ifdef SHARED
            const int w = 0;
#else
            const int w = q;
#endif
            for (int k = 0; k < nwin; ++k) {
                if (k == 0)                      // the writer reads before it writes
                    wrong += mgb::list_start(tb.data(), w, nseg, (int)((window + 2) % 3)) != base - before;
                mgb::set_list_start(tb.data(), w, nseg, (int)((window + k) % 3), base + (int64_t)k * nst);
                if (k == std::min(ahead, nwin - 1))
                    wrong += mgb::list_start(tb.data(), w, nseg, (int)((window + 2) % 3)) != base - before;
            }
        }
        base += (int64_t)nwin * nst;
        window += nwin;
        before = nst;
    }
#ifndef SHARED
    for (int q = 0; q < nseg; ++q)               // between runs: the same in every segment
        for (int b = 0; b < 3; ++b) wrong += tb[b * nseg + q] != tb[b * nseg];
#endif
    return wrong;
}
int main() {
    int wrong = 0, n = 0;
    for (int nseg = 1; nseg <= 4; ++nseg) {
        std::vector<int> order(nseg);
        std::iota(order.begin(), order.end(), 0);
        do {
            for (int nwin = 1; nwin <= 7; ++nwin)
                for (int rest = 0; rest <= 2; ++rest)        // windows of other lengths between the launches
                    for (int ahead = 0; ahead <= 1; ++ahead) {
                        std::vector<std::pair<int, int>> l;
                        for (int r = 0; r < 4; ++r) {
                            l.push_back({nwin, 10});
                            for (int k = 0; k < rest; ++k) l.push_back({1, 3 + k});
                        }
                        wrong += run(nseg, l, order, ahead);
                        ++n;
                    }
        } while (std::next_permutation(order.begin(), order.end()));
    }
    std::printf("%d launches' orders, %d wrong starts\n", n, wrong);
    return wrong ? 1 : 0;
}
"""


@pytest.mark.parametrize("shared", [False, True])
def test_starts_with_segments_apart(tmp_path, shared):
    """Words of each segment's own: every start right.  One set of words for all segments
    (the model's own mistake): the model sees it."""
    src, exe = tmp_path / "model.cpp", tmp_path / "model"
    src.write_text(MODEL)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "mgbrain_amd", "csrc"), *(["-DSHARED"] if shared else []),
                    "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == (1 if shared else 0), r.stdout
