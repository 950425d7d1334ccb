// BFS and SSSP levels as a team runs them (team.h).
//
// A wave takes TEAM_PIECE records of one member at a time, a lane per edge, one or two
// pieces in step.  After a meeting every wave knows all members' counts and finds its pieces
// by itself.
#pragma once

#include <climits>

#include "team.h"

namespace mg {

// BFS: the neighbour id, then its claim (test-and-set of the visited bit) and its offsets
// together, so a claimed vertex joins the next frontier as records of its edge range and
// the next level starts at the adjacency.  Runs from meeting `it` (posted, frontier L) until
// stop(words) says so; it is asked at every meeting, by every wave alike.  HUB: TeamCtl::hub is
// set where that is why a member overflows (in the posts it cost the single searches 0.6%).
// Bound by the chain record -> neighbour -> claim / offsets -> post -> meeting, about 3 us
// at 1000 vertices a level.  2048^2 grid: 15.6 ms when first written like this, 20.9 ms with
// a lane per record (four edges each) and workgroup-wide queues; 8 workgroups 22 ms; one /
// four pieces in step 16.6 / 15.6 ms.
template <bool HUB = false, class Stop>
__device__ __forceinline__ void team_bfs(const TeamSeat &t, const int *off, const int *adj, uint32_t *visited,
                                         int *depth, int &L, int &it, Stop stop) {
    const int sub = lane_id() % TEAM_EDGES;
    for (;; ++it) {
        const uint64_t w = team_meet(t.ctl, it, t.size);
        const TeamIn in = team_in(t.recs, it, w);
        if (stop(w)) return;
        TeamOut out(t.recs, it + 1, t.rank);
        // K pieces in step, each stage's accesses in flight together
        auto expand = [&](auto kc, int p0) {
            constexpr int K = decltype(kc)::value;
            uint64_t rec[K];
            int u[K];
            bool on[K];
            uint32_t old[K];
            IntPair o[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                on[k] = true;
                rec[k] = team_fetch(in, p0 + k * t.size, on[k]);
            }
#pragma unroll
            for (int k = 0; k < K; ++k) {
                on[k] = on[k] && sub < rec_len(rec[k]);
                u[k] = adj[rec_beg(rec[k]) + (on[k] ? sub : 0)];
            }
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (on[k])
                    old[k] = __hip_atomic_fetch_or(&visited[u[k] >> 5], 1u << (u[k] & 31), __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int k = 0; k < K; ++k) o[k] = ld_range(off, u[k]);
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const bool first = on[k] ? !((old[k] >> (u[k] & 31)) & 1u) : false;
                const uint64_t firsts = wave_ballot(first);
                if (!firsts) continue;
                if (first) depth[u[k]] = L + 1;
                out.queue(first, firsts, 0, o[k]);
            }
        };
        int p = t.rank;
        for (; p + t.size < in.pieces; p += 2 * t.size) expand(std::integral_constant<int, 2>(), p);
        if (p < in.pieces) expand(std::integral_constant<int, 1>(), p);
        ++L;
        if (HUB && out.hub) team_set_hub(t.ctl);
        team_post(t.ctl, it + 1, t.rank, out.word(it + 1));
    }
}

// SSSP: neighbour and weight with the vertex's distance, then the neighbour's distance and
// offsets, then for a candidate the minimum and the claim together (a stale, larger
// distance only causes a redundant relaxation).  Claims are test-and-sets: below the
// bucket bound in the next level's frontier bitmap (the winner queues the vertex), else in
// the far bitmap, which is the whole far list.  Whoever takes a vertex clears its frontier
// bit, so the bitmaps rotate clean and always hold the frontier (vertices without
// out-edges aside, which need no relaxing).  When no record is left the members move the
// bound and sweep the far bitmap (n bits: about 1 us at 1M vertices, once per bucket).
struct TeamSssp {
    const int *off, *adj, *w;
    int *dist;
    uint32_t *bm0, *bm1, *bm2, *farbm;  // frontier bitmaps (level L: bm0, bm1, bm2 by L % 3), far bitmap
    int nwords, limit;
    long long delta, thr, unbucketed;  // no distance reaches a bound of `unbucketed`
    long long ex = 0;                  // edges this lane relaxed
};

// Runs from meeting `it` (posted, frontier L) until the search ends or reaches its level
// limit (true), or until a member overflows or wide(words) says so (false; bitmap
// L % 3 then holds the frontier).  closed(words) is called after each level.
template <bool HUB = false, class Closed, class Wide>
__device__ __forceinline__ bool team_sssp(const TeamSeat &t, TeamSssp &s, int &L, int &it, Closed closed, Wide wide) {
    const int lane = lane_id(), sub = lane % TEAM_EDGES;
    // (locals: with its fields read in place the struct stayed in scratch memory)
    const int *const off = s.off, *const adj = s.adj, *const wts = s.w;
    int *const dist = s.dist;
    uint32_t *const b0 = s.bm0, *const b1 = s.bm1, *const b2 = s.bm2, *const farbm = s.farbm;
    const int nwords = s.nwords, limit = s.limit;
    const long long delta = s.delta, unbucketed = s.unbucketed;
    long long thr = s.thr, ex = 0;
    bool swept = false, done = false;  // swept: this meeting's records come from the far bitmap
    auto bitmap = [&](int l) { return l % 3 == 0 ? b0 : l % 3 == 1 ? b1 : b2; };
    for (;; ++it) {
        const uint64_t w = team_meet(t.ctl, it, t.size);
        const TeamIn in = team_in(t.recs, it, w);
        long long sweep_from = -1;  // >= 0: sweep, dropping waiting distances below this
        // the same decisions in every wave
        if (wave_ballot(team_over(w)) != 0) break;
        if (!swept) closed(w);
        if (L >= limit) {
            done = true;
        } else if (in.pieces > 0) {
            if (wide(w)) break;
        } else if (thr >= unbucketed) {
            done = true;
        } else if (!swept) {
            sweep_from = thr;
            thr += delta;
        } else {
            // nothing waits in that bucket: the one of the smallest waiting distance
            int lo = lane < t.size ? ld_dev(&t.ctl->least[it & 1][lane]) : INT_MAX;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) lo = min(lo, __shfl_xor(lo, o));
            if (lo == INT_MAX) {
                done = true;
            } else {
                sweep_from = thr;
                thr = ((long long)lo / delta + 1) * delta;
            }
        }
        if (done) break;
        TeamOut out(t.recs, it + 1, t.rank);
        swept = sweep_from >= 0;
        if (swept) {
            // far vertices below the bound join frontier L (its bitmap is clear); those
            // below the old bound were relaxed since and leave the far bitmap
            uint32_t *fr = bitmap(L);
            int least = INT_MAX;
            team_words(farbm, nwords, t.rank, t.size, [&](int i, uint32_t word) {
                uint32_t todo = word, keep = 0, go = 0;
                while (wave_ballot(todo != 0)) {
                    const bool has = todo != 0;
                    const int b = has ? __ffs(todo) - 1 : 0, u = has ? i * 32 + b : 0;
                    todo &= todo - 1;
                    const int d = ld_dev(&dist[u]);
                    const IntPair o = ld_range(off, u);
                    const bool take = has && d >= sweep_from && d < thr && o.b > o.a;
                    if (has && d >= thr) {
                        keep |= 1u << b;
                        least = min(least, d);
                    }
                    if (take) go |= 1u << b;
                    const uint64_t takes = wave_ballot(take);
                    if (takes) out.queue(take, takes, u, o);
                }
                if (keep != word) __hip_atomic_store(&farbm[i], keep, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                if (go) __hip_atomic_store(&fr[i], go, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            });
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) least = min(least, __shfl_xor(least, o));
            if (lane == 0)
                __hip_atomic_store(&t.ctl->least[(it + 1) & 1][t.rank], least, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
            if (HUB && out.hub) team_set_hub(t.ctl);
            team_post(t.ctl, it + 1, t.rank, out.word(it + 1));
            continue;
        }
        uint32_t *fr = bitmap(L), *nx = bitmap(L + 1);
        auto relax = [&](auto kc, int p0) {
            constexpr int K = decltype(kc)::value;
            uint64_t rec[K];
            int u[K], wt[K], dv[K], du[K];
            bool on[K];
            IntPair o[K];
            uint32_t old[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                on[k] = true;
                rec[k] = team_fetch(in, p0 + k * t.size, on[k]);
            }
#pragma unroll
            for (int k = 0; k < K; ++k) {
                on[k] = on[k] && sub < rec_len(rec[k]);
                const int e = rec_beg(rec[k]) + (on[k] ? sub : 0);
                u[k] = adj[e];
                wt[k] = wts[e];
                dv[k] = ld_dev(&dist[rec_vertex(rec[k])]);
            }
#pragma unroll
            for (int k = 0; k < K; ++k) {
                du[k] = ld_dev(&dist[u[k]]);
                o[k] = ld_range(off, u[k]);
                if (on[k] && sub == 0)
                    __hip_atomic_store(&fr[rec_vertex(rec[k]) >> 5], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            bool cand[K], near[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const long long nd = (long long)dv[k] + wt[k];
                ex += on[k];
                cand[k] = on[k] && nd < du[k];
                near[k] = nd < thr;
                if (cand[k]) {
                    __hip_atomic_fetch_min(&dist[u[k]], (int)nd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    old[k] = __hip_atomic_fetch_or(&(near[k] ? nx : farbm)[u[k] >> 5], 1u << (u[k] & 31),
                                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
#pragma unroll
            for (int k = 0; k < K; ++k) {
                bool first = cand[k] && near[k] ? !((old[k] >> (u[k] & 31)) & 1u) : false;
                // a vertex without out-edges has no record to clear its bit
                if (first && o[k].a == o[k].b) {
                    __hip_atomic_fetch_and(&nx[u[k] >> 5], ~(1u << (u[k] & 31)), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
                    first = false;
                }
                const uint64_t firsts = wave_ballot(first);
                if (firsts) out.queue(first, firsts, u[k], o[k]);
            }
        };
        int p = t.rank;
        for (; p + t.size < in.pieces; p += 2 * t.size) relax(std::integral_constant<int, 2>(), p);
        if (p < in.pieces) relax(std::integral_constant<int, 1>(), p);
        ++L;
        if (HUB && out.hub) team_set_hub(t.ctl);
        team_post(t.ctl, it + 1, t.rank, out.word(it + 1));
    }
    s.thr = thr;
    s.ex += ex;
    return done;
}

}  // namespace mg
