// Rules of the host side that need no device code (so they are tested without a GPU).
#pragma once

#include <cstdint>

#include "mg_internal.h"

namespace mg {

// Kinds of captured steps a graph keeps, one executable graph each.
enum { KIND_BFS = 0, KIND_SSSP = 1, KIND_PR = 2, KIND_GAS = 3, KIND_BATCH = 4, KIND_BATCH_SSSP = 5, KIND_BATCH_PULL = 6, NKINDS = 8 };

// What a batched search's captured steps are kept under.  Two routes whose steps work on
// different state never share one: a search that found the other route's steps would replay
// them and wait for a control block that they do not touch.
struct StepKey {
    int kind;
    uint64_t key;
};
inline StepKey batch_sssp_steps(long long delta) { return {KIND_BATCH_SSSP, mix64((uint64_t)delta)}; }
inline StepKey batch_pull_steps(int k) { return {KIND_BATCH_PULL, (uint64_t)k}; }

}  // namespace mg
