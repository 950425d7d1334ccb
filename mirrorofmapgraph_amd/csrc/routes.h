// Rules of the host side that need no device code (so they are tested without a GPU).
#pragma once

#include <cstdint>

#include "mg_internal.h"

namespace mg {

// Kinds of captured steps a graph keeps, one executable graph each (KIND_BATCH_PULL: four, by
// row width).
enum { KIND_BFS = 0, KIND_SSSP = 1, KIND_PR = 2, KIND_GAS = 3, KIND_BATCH = 4, KIND_BATCH_SSSP = 5, KIND_BATCH_PULL = 6, NKINDS = 10 };

// What a batched search's captured steps are kept under.  Two routes whose steps work on
// different state never share one: a search that found the other route's steps would replay
// them and wait for a control block that they do not touch.
struct StepKey {
    int kind;
    uint64_t key;
};
inline StepKey batch_sssp_steps(long long delta) { return {KIND_BATCH_SSSP, mix64((uint64_t)delta)}; }
// Pulled rows: 32, 64, 128 or 256 distances a vertex, four a lane.  k itself is read from
// device memory, so calls of any sizes replay the rounds of their width: keyed on k, a caller
// whose batches vary captured them again on each call (R-MAT scale 16, 17 to 28 sources: 968
// us a call, 796 with k fixed).
inline int pull_width(int k) { return k <= 32 ? 0 : k <= 64 ? 1 : k <= 128 ? 2 : 3; }
inline int pull_lanes(int k) { return 8 << pull_width(k); }
inline StepKey batch_pull_steps(int k) { return {KIND_BATCH_PULL + pull_width(k), 0}; }

// Narrow levels in a row that the single workgroup runs before a team takes over (team.h): at
// first, after a team that ran `levels` levels when it was asked for after `after`, and at the
// start of the graph's next search.  The hand-over and the way back cost some ten levels of
// the single workgroup (the steps queued behind the pause, a wait of the host, the frontier
// rebuilt from the depths), so a team that soon outgrows its queues or meets a hub has to be
// waited for four times as long.  Asking again after a single narrow level, searches that
// alternate took up to nine times as long as without teams (300 stars of 1100 leaves on a
// path: SSSP 9.4 -> 82 ms, so 9.6).
constexpr int TEAM_AFTER = 8;
constexpr int team_after_next(int after, int levels) {
    return levels >= 4 * TEAM_AFTER || after >= 1 << 20 ? after : 4 * after;
}
constexpr int team_after_start(int last) { return last / 4 > TEAM_AFTER ? last / 4 : TEAM_AFTER; }

// How a launch of teams ended (TeamsCtl::end, the largest of its rows').
enum {
    TEAMS_DONE = 0,
    TEAMS_SHORT = 1,     // a row outgrew a team of fewer workgroups than it was to have (a busy GPU)
    TEAMS_OUTGROWN = 2,  // a row outgrew a whole team
    TEAMS_HUB = 3,       // a row reached a vertex of more out-edges than a team queues
};

// What a graph's batched searches of one kind found out about teams.
struct TeamsRule {
    int wgs = 0;        // least workgroups of a team, since smaller ones were outgrown (0: none yet)
    int skip = 0;       // calls to come that don't try
    int wait = 0;       // how many the last failure made it

    // Whether this call tries (called once a call).
    bool wanted() {
        if (skip == 0) return true;
        --skip;
        return false;
    }
    // After a launch of teams of `wgs_now` workgroups that ended short of its rows: whether to
    // run the call again by teams, else the general route takes it.  A larger team helps only
    // where a whole one was outgrown; a short one says nothing about the graph, and gets one
    // more try (`again`: it had that).  A failure that belongs to the graph and the sources is
    // not repeated at once: the next 32 calls, then 128, 512, ... don't try.
    bool retry(int end, int wgs_now, int wgs_most, bool again) {
        if (end == TEAMS_SHORT) return !again;
        if (end == TEAMS_OUTGROWN && wgs_now < wgs_most) {
            wgs = 2 * wgs_now;
            return true;
        }
        wait = wait == 0 ? 32 : wait < 1 << 20 ? 4 * wait : wait;
        skip = wait;
        return false;
    }
    void succeeded() { wait = 0; }
};

// When an idle personalized PageRank engine of a server starts a cohort: at `batch` waiting
// queries, or when the oldest has waited `us`.  Values given in the configuration count as
// they are.  By default a server that is busy (PPR_BUSY queries of other engines running or
// waiting) waits longer for larger cohorts: the sweeps otherwise end sooner, start again for
// fewer queries and keep the memory as busy (benchmark mix of 2000 queries a second, some 110
// outstanding, 20 ms and 8 queries / 70 ms and 16: median of all queries 74 / 39 ms, 99th
// percentile 440 / 330).  On one that is not, the wait is all that a query notices: at 100
// queries a second, where a single running query had lengthened the gate, R-MAT scale 16 took
// 72 ms a query instead of 24.
constexpr int PPR_BUSY = 64;
struct PprGate {
    int batch, us;
};
inline PprGate ppr_gate(int cfg_us, int cfg_batch, int64_t others) {
    const bool busy = others >= PPR_BUSY;
    return {cfg_batch > 0 ? cfg_batch : busy ? 16 : 8, cfg_us > 0 ? cfg_us : busy ? 70000 : 20000};
}

}  // namespace mg
