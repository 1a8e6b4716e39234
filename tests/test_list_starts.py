"""Which window wrote a spike list (csrc/mgb_lists.h), in a CPU model of runs whose
segments are windows apart: each segment's workgroups wait only for their own segment, so
one segment may have ended a persistent launch before another's first workgroup has read
the words that the run before left."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MODEL = r"""
#include <algorithm>
#include <cstdio>
#include <numeric>
#include <vector>
#include "mgb_lists.h"
// Runs of `steps` steps in windows of `window`, as the host issues them: the whole windows in
// one persistent launch (or each in its own), then the rest.  The segments of a launch go
// one after another in `order`, each through all its windows.  SHARED: segment 0 writes every
// window's start into the words (the model's own mistake).
static int runs(const std::vector<int>& lengths, int window, bool persistent, const std::vector<int>& order) {
    int64_t tb[3] = {0, 0, 0}, base = 0, win = 0, before = 0;   // before: steps of the last window issued
    int wrong = 0;
    for (int steps : lengths) {
        int off = 0, wk = 0, prev = 0;
        const int whole = steps / window;
        auto launch = [&](int nwin, int nst) {
            for (int q : order) {
                const int64_t s0 = base + off;
                wrong += mgb::window_before(tb, mgb::mod3(win + wk + 2), s0, prev) != s0 - before;
#ifdef SHARED
                if (q == 0)
                    for (int k = 0; k < nwin; ++k) tb[(win + wk + k) % 3] = s0 + (int64_t)k * nst;
#endif
            }
            off += nwin * nst;
            wk += nwin;
            before = prev = nst;
        };
        if (persistent && whole >= 2) launch(whole, window);
        while (off < steps) launch(1, std::min(window, steps - off));
        mgb::end_run(tb, base, win, steps, wk, prev);
        base += steps;
        win += wk;
    }
    return wrong;
}
int main() {
    int wrong = 0, n = 0;
    for (int64_t k = 0; k < 1000; ++k)
        for (int64_t at : {(int64_t)0, ((int64_t)1 << 32) - 500, ((int64_t)1 << 40) + 7, (int64_t)0x7FFFFFFFFFFFF000})
            wrong += mgb::mod3(at + k) != (int)((at + k) % 3);
    for (int nseg = 1; nseg <= 4; ++nseg) {
        std::vector<int> order(nseg);
        std::iota(order.begin(), order.end(), 0);
        do
            for (int window : {1, 3, 10})
                for (int a = 1; a <= 75; a += 2)
                    for (int b = 1; b <= 40; b += 3)
                        for (bool p : {true, false}) {
                            wrong += runs({a, b, a, a, b}, window, p, order);
                            ++n;
                        }
        while (std::next_permutation(order.begin(), order.end()));
    }
    std::printf("%d models, %d wrong starts\n", n, wrong);
    return wrong ? 1 : 0;
}
"""


@pytest.mark.parametrize("shared", [False, True])
def test_starts_with_segments_apart(tmp_path, shared):
    """Every start is the one of the window before, in whatever order the segments run; with
    the words written during a launch the model sees wrong ones."""
    src, exe = tmp_path / "model.cpp", tmp_path / "model"
    src.write_text(MODEL)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "mgbrain_amd", "csrc"),
                    *(["-DSHARED"] if shared else []), "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == (1 if shared else 0), r.stdout
