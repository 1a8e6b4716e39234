// mgb_lists.h -- start steps of the fused path's spike lists, shared by the kernels, the
// host and a CPU model of a launch.
//
// A window's propagation needs the first step of the window before it, whose list it
// reads.  Inside a persistent launch that is the launch's own window length; in a launch's
// first window it is the word that the previous launch left.  The words are [3][nseg], one
// per list and segment: a segment's workgroups wait only for each other between windows, so
// another segment can be any number of windows ahead while one of this segment has yet to
// start, and would have written over a word they shared (window k + 2 goes to the list of
// window k - 1).  In its own segment no workgroup is more than one window ahead of the
// last, and window k + 1 writes neither list k nor list k - 1.
#pragma once
#include <stdint.h>

#include "mgb_rng.h"

namespace mgb {

// First step of the window that wrote list b (0, 1, 2) of segment q.  All three words load,
// then b picks one: b comes from a load of its own.
MGB_HD int64_t list_start(const int64_t* tbase, int32_t q, int32_t nseg, int b) {
    const int64_t s0 = tbase[q], s1 = tbase[nseg + q], s2 = tbase[2 * nseg + q];
    return b == 0 ? s0 : (b == 1 ? s1 : s2);
}

// (by one workgroup of segment q)
MGB_HD void set_list_start(int64_t* tbase, int32_t q, int32_t nseg, int b, int64_t step) {
    tbase[b * nseg + q] = step;
}

}  // namespace mgb
