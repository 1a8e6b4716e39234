// mgb_lists.h -- which window wrote a spike list of the fused path, shared by the kernels
// and a CPU model of a run's launches.
//
// A window's propagation needs the first step of the window before it, whose list it reads:
// the window's own length inside a persistent launch, the length that the host gives with
// each later launch of a run, and in a run's first launch a word (one per list) that the
// run before left.  Only the end of a run writes these words.  No launch does: a segment's
// workgroups wait only for each other between windows, so that another segment can be any
// number of windows ahead while one of this segment has yet to read them.
#pragma once
#include <stdint.h>

#include "mgb_rng.h"

namespace mgb {

// The list of window k (>= 0): k mod 3 in 32-bit arithmetic (2^32 = 1 mod 3; the 64-bit
// remainder takes well over a hundred instructions on the device).
MGB_HD int mod3(int64_t k) {
    return (int)(((uint32_t)((uint64_t)k >> 32) % 3u + (uint32_t)k % 3u) % 3u);
}

// First step of the window before the one that starts at s0, whose list is b (0, 1, 2), in
// the first window of a launch: prev_len steps earlier, or (0) by the words.  All three load,
// then b picks one: b comes from a load of its own.
MGB_HD int64_t window_before(const int64_t* tbase, int b, int64_t s0, int32_t prev_len) {
    if (prev_len) return s0 - prev_len;
    const int64_t t0 = tbase[0], t1 = tbase[1], t2 = tbase[2];
    return b == 0 ? t0 : (b == 1 ? t1 : t2);
}

// End of a run of `steps` steps in `windows` windows (at least one) from base_step and
// base_window on, whose last window had `last` steps.
MGB_HD void end_run(int64_t* tbase, int64_t base_step, int64_t base_window, int32_t steps, int32_t windows,
                    int32_t last) {
    tbase[mod3(base_window + windows - 1)] = base_step + steps - last;
}

}  // namespace mgb
