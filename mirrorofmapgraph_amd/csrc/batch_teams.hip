// Batched searches as single-source searches side by side, a team of waves each
// (team_search.h): the path of mg_bfs_batch / mg_sssp_batch on sparse graphs (meshes),
// whose searches are hundreds or thousands of narrow levels.
//
// The shared-frontier batches (batch.hip, batch_sssp.hip) take four or five launches per
// level for all sources together, whatever little the level holds: 64 SSSP sources on a
// 512^2 grid are 1850 rounds of about 10,000 (vertex, source) pairs, 41 us each.  Here up to
// TEAMS_MAX teams take rows from a counter and run each to its end in one launch, the
// level boundary being a meeting of the team (about 1 us); a row is the team's depth or
// distance array itself.  The teams share TEAMS_GRID workgroups.  A row whose frontier
// outgrows a team's queues says why in TeamsCtl::end, every team stops at its next row and
// the call is run again, by larger teams or the shared way (TeamsRule).
//
// Bound by each team's chain of accesses and meetings, 4 to 5 us a level with 64 teams.
// 64 SSSP sources on a 512^2 grid 76 -> 6.0 ms (93 before the shared batches' slices fitted
// the grid); with 1024 workgroups 6.4 ms.  256 sources: SSSP 13.8 ms with 256 teams of two
// workgroups, 17.8 with 128 of eight, 24 with 64 of 16; BFS 11.3 / 12.2 / 13.8 ms.
#include <cmath>
#include <cstdlib>

#include "batch.h"
#include "team_search.h"

namespace mg {

constexpr int TEAMS_GRID = 512;  // workgroups of the teams together: two per CU
constexpr int TEAMS_MAX = 256;   // teams
constexpr int XCDS = 8;
// Sparse: fewer edges than this per vertex.  The same line as mg_bfs_batch's levels: a
// search of a denser graph has a wide level soon, and would only be started for nothing.
constexpr int64_t TEAMS_DEGREE = 8;
// A level of a mesh has up to a few times sqrt(n) vertices (buckets: twice that): teams are
// given room for TEAMS_FRONT (SSSP 2 x) sqrt(n) records, which many small ones lack on a
// large graph, and twice the workgroups, down to 32 teams of 16, when a row outgrows one all
// the same.  2048^2 grid, 256 rows (two workgroups a team outgrown, the call run again in
// general / so): BFS 410 / 159 ms, SSSP 884 / 284; on the 512^2 grid two workgroups do.
constexpr int TEAMS_FRONT = 4;
// State kept when the route is given up for a while: freeing what kernels have used takes 0.5
// ms, half of a small call (one source on a random graph of 100,000 vertices: first call 1.63
// ms so, 1.07 kept), and the next try would make it again.  Larger ones are released.
constexpr int64_t TEAMS_KEEP = 64LL << 20;

struct TeamsCtl {
    int arrived[16];             // workgroups that came, by XCD
    int next, end, levels, pad;  // next row; TEAMS_DONE or why a row ended (no team takes another then); most levels of a row
    unsigned long long edges, te, nr;  // edges relaxed; TEPS count and reached vertices
};

// Device state of a graph's team batches: one block, laid out anew by each call (nothing in it
// outlives one).
struct TeamsDev {
    char *block = nullptr;
    int64_t cap = 0;
};

struct TeamsArgs {
    TeamsCtl *ctl;
    TeamCtl *team;
    uint64_t *recs;
    uint32_t *bits;
    int *rows;
    const int *row_start, *srcs;
    const int *off, *adj, *w;
    int n, nwords, k, per_xcd, wgs, limit;
    long long delta;
};

// Unreached rows, empty bitmaps and open teams.
__global__ void teams_init(TeamsArgs a, int unreached) {
    const int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, nt = (int64_t)gridDim.x * blockDim.x;
    const int64_t total = (int64_t)a.k * a.n;
    if (((uintptr_t)a.rows & 15) == 0) {
        int4 *r4 = reinterpret_cast<int4 *>(a.rows);
        for (int64_t i = tid; i < total / 4; i += nt) r4[i] = make_int4(unreached, unreached, unreached, unreached);
        for (int64_t i = total / 4 * 4 + tid; i < total; i += nt) a.rows[i] = unreached;
    } else {
        for (int64_t i = tid; i < total; i += nt) a.rows[i] = unreached;
    }
    const int teams = XCDS * a.per_xcd;
    for (int64_t i = tid; i < 4LL * teams * a.nwords; i += nt) a.bits[i] = 0;
    int *t = reinterpret_cast<int *>(a.team);
    for (int64_t i = tid; i < (int64_t)(sizeof(TeamCtl) / 4) * teams; i += nt) t[i] = 0;
    int *c = reinterpret_cast<int *>(a.ctl);
    for (int64_t i = tid; i < (int64_t)(sizeof(TeamsCtl) / 4); i += nt) c[i] = 0;
}

// The whole workgroup joins the next team of its XCD; false when that has enough.
__device__ __forceinline__ bool teams_join(const TeamsArgs &a, int &team, TeamSeat &t) {
    __shared__ int s_team;
    if (threadIdx.x == 0) {
        const int x = xcd_id() % XCDS;
        const int q = atomicAdd(&a.ctl->arrived[x], 1) / a.wgs;
        s_team = q < a.per_xcd ? x * a.per_xcd + q : -1;
    }
    __syncthreads();
    team = s_team;
    if (team < 0) return false;
    t.ctl = a.team + team;
    t.recs = a.recs + (size_t)team * TEAM_RECS;
    return team_join(t.ctl, a.wgs, t.rank, t.size);
}

// Clears this wave's share of a bitmap.
__device__ __forceinline__ void teams_clear(uint32_t *bm, int nwords, const TeamSeat &t) {
    for (int i = t.rank * WAVE + lane_id(); i < nwords; i += t.size * WAVE)
        __hip_atomic_store(&bm[i], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Starts the team's next row: member 0 takes it from the counter and seeds its sources
// (bits of `seen`, value 0, records).  Every wave returns the row, or -1 when none is
// left; `it` is the meeting with the row's first records.  The meeting before it ends
// the previous row for every member, bitmaps cleared.
template <bool EDGES>
__device__ __forceinline__ int teams_next(const TeamsArgs &a, const TeamSeat &t, uint32_t *seen, int &it) {
    const int lane = lane_id();
    ++it;
    team_post(t.ctl, it, t.rank, team_word(it, false, 0, 0, 0));
    team_meet(t.ctl, it, t.size);
    ++it;
    uint64_t word = team_word(it, false, 0, 0, 0);
    if (t.rank == 0) {
        int row = 0;
        if (lane == 0) row = ld_dev(&a.ctl->end) ? a.k : atomicAdd(&a.ctl->next, 1);
        row = __builtin_amdgcn_readfirstlane(row);
        if (row < a.k) {
            TeamOut out(t.recs, it, 0);
            const int end = a.row_start[row + 1];
            for (int i0 = a.row_start[row]; i0 < end; i0 += WAVE) {
                const bool has = i0 + lane < end;
                const int v = a.srcs[has ? i0 + lane : i0];
                const IntPair o = ld_range(a.off, v);
                if (has) a.rows[(int64_t)row * a.n + v] = 0;
                // SSSP: a vertex without out-edges has no record to clear its bit
                bool first = has && (!EDGES || o.b > o.a);
                uint32_t old = 0;
                if (first)
                    old = __hip_atomic_fetch_or(&seen[v >> 5], 1u << (v & 31), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                first = first && !((old >> (v & 31)) & 1u);
                const uint64_t firsts = wave_ballot(first);
                if (firsts) out.queue(first, firsts, v, o);
            }
            // the out-edges' field carries the row
            if (out.hub) team_set_hub(t.ctl);
            word = team_over(out.word(it)) ? team_word(it, true, 0, 0, row + 1)
                                           : team_word(it, false, out.nrec, min(out.nf, 0xffff), row + 1);
        }
    }
    team_post(t.ctl, it, t.rank, word);
    const uint64_t w = team_meet(t.ctl, it, t.size);
    const uint32_t low = __builtin_amdgcn_readfirstlane((uint32_t)w);  // member 0's
    return (int)(low & 0xfffff) - 1;
}

__device__ __forceinline__ void teams_row_done(const TeamsArgs &a, const TeamSeat &t, int L, bool over) {
    if (t.rank != 0 || lane_id() != 0) return;
    atomicMax(&a.ctl->levels, L);
    if (over) atomicMax(&a.ctl->end, ld_dev(&t.ctl->hub) ? TEAMS_HUB : t.size < a.wgs * (BLK / WAVE) ? TEAMS_SHORT : TEAMS_OUTGROWN);
}

__global__ __launch_bounds__(BLK) void teams_bfs(TeamsArgs a) {
    int team, it = 0;
    TeamSeat t;
    if (!teams_join(a, team, t)) return;
    uint32_t *visited = a.bits + (size_t)team * 4 * a.nwords;
    for (;;) {
        const int row = teams_next<false>(a, t, visited, it);
        if (row < 0) return;
        int L = 0;
        bool over = false;
        team_bfs<true>(t, a.off, a.adj, visited, a.rows + (int64_t)row * a.n, L, it, [&](uint64_t w) {
            over = wave_ballot(team_over(w)) != 0;
            return over || wave_ballot(team_nf(w) != 0) == 0 || L >= a.limit;
        });
        teams_row_done(a, t, L, over);
        if (!over) teams_clear(visited, a.nwords, t);
    }
}

__global__ __launch_bounds__(BLK) void teams_sssp(TeamsArgs a) {
    int team, it = 0;
    TeamSeat t;
    if (!teams_join(a, team, t)) return;
    TeamSssp s;
    s.off = a.off;
    s.adj = a.adj;
    s.w = a.w;
    s.bm0 = a.bits + (size_t)team * 4 * a.nwords;
    s.bm1 = s.bm0 + a.nwords;
    s.bm2 = s.bm1 + a.nwords;
    s.farbm = s.bm2 + a.nwords;
    s.nwords = a.nwords;
    s.limit = a.limit;
    s.delta = a.delta;
    s.unbucketed = LLONG_MAX / 4;
    for (;;) {
        const int row = teams_next<true>(a, t, s.bm0, it);
        if (row < 0) break;
        s.dist = a.rows + (int64_t)row * a.n;
        s.thr = a.delta;
        int L = 0;
        const bool done = team_sssp<true>(t, s, L, it, [](uint64_t) {}, [](uint64_t) { return false; });
        teams_row_done(a, t, L, !done);
        if (done && L >= a.limit) {  // stopped short: the frontier and the far vertices are left
            teams_clear(s.bm0, a.nwords, t);
            teams_clear(s.bm1, a.nwords, t);
            teams_clear(s.bm2, a.nwords, t);
            teams_clear(s.farbm, a.nwords, t);
        }
    }
    const long long ex = wave_sum_ll(s.ex);
    if (lane_id() == 0) atomicAdd(&a.ctl->edges, (unsigned long long)ex);
}

// TEPS count and reached vertices of the rows (grid: x over vertices, y over rows).
__global__ __launch_bounds__(BLK) void teams_stats(TeamsArgs a, int unreached) {
    const int *row = a.rows + (int64_t)blockIdx.y * a.n;
    long long te = 0, nr = 0;
    for (int v = blockIdx.x * BLK + (int)threadIdx.x; v < a.n; v += gridDim.x * BLK)
        if (row[v] != unreached) {
            ++nr;
            te += a.off[v + 1] - a.off[v];
        }
    te = block_sum<BLK>(te);
    nr = block_sum<BLK>(nr);
    if (threadIdx.x == 0) {
        atomicAdd(&a.ctl->te, (unsigned long long)te);
        atomicAdd(&a.ctl->nr, (unsigned long long)nr);
    }
}

// ---------------------------------------------------------------- host side

void teams_release(mg_graph *g) {
    TeamsDev *&t = g->steps->teams;
    if (!t) return;
    free_dev(t->block);
    delete t;
    t = nullptr;
    g->steps->teams_bytes = 0;
}

// Workgroups launched for a team of wgs; fewer with MG_TEAM_LAUNCH in the environment, for
// tests of teams that close short, as on a busy GPU.
static int teams_launch(int wgs) {
    const char *e = getenv("MG_TEAM_LAUNCH");
    return e && *e ? std::clamp(atoi(e), 1, wgs) : wgs;
}

// Runs the call; *end says whether its rows were finished (else nothing is delivered) and
// *wgs how many workgroups a team was to have.
static int teams_batch(mg_graph *g, bool sssp, const int32_t *row_of, const int32_t *srcs, int32_t npairs, int32_t k,
                       int32_t *out, const mg_options &o, mg_stats *stats, const CallTimer &timer, int *end, int *wgs) {
    TeamsDev *&tp = g->steps->teams;
    if (!tp && !(tp = new (std::nothrow) TeamsDev())) return set_error(MG_ERR_OOM, "host allocation failed");
    TeamsDev &t = *tp;
    const int nwords = ((g->n + 63) / 64) * 2;
    const int room = TEAM_SEG * (BLK / WAVE);  // records a workgroup queues
    const int front = (int)std::min(1e6, (sssp ? 2 : 1) * TEAMS_FRONT * std::sqrt((double)g->n));
    const int least = std::min(TEAM_WGS, std::max(g->steps->teams_rule[sssp].wgs, (front + room - 1) / room));
    const int per_xcd = std::min({(k + XCDS - 1) / XCDS, TEAMS_MAX / XCDS, TEAMS_GRID / XCDS / least}), teams = per_xcd * XCDS;
    // the sources by row
    std::vector<int32_t> pairs((size_t)MG_BATCH_MAX + 1 + (size_t)npairs, 0);
    int32_t *start = pairs.data(), *list = start + MG_BATCH_MAX + 1;
    for (int i = 0; i < npairs; ++i) start[row_of[i] + 1]++;
    for (int r = 0; r < k; ++r) start[r + 1] += start[r];
    {
        std::vector<int32_t> at(start, start + k);
        for (int i = 0; i < npairs; ++i) list[at[(size_t)row_of[i]]++] = srcs[i];
    }
    const int64_t cells = (int64_t)k * g->n;
    const bool direct = plan_delivery(g, out, 4 * (size_t)cells, o.out_on_device).as_state;
    int64_t need = 0;
    auto part = [&](int64_t bytes) {
        const int64_t at = need;
        need += (bytes + 4095) / 4096 * 4096;
        return at;
    };
    const int64_t at_ctl = part(sizeof(TeamsCtl)), at_pairs = part(4 * (int64_t)pairs.size()),
                  at_team = part(teams * (int64_t)sizeof(TeamCtl)), at_recs = part(teams * 8 * (int64_t)TEAM_RECS),
                  at_bits = part(teams * 16 * (int64_t)nwords), at_rows = part(direct ? 0 : 4 * cells);
    if (t.cap < need) {
        free_dev(t.block);
        t.block = nullptr;
        t.cap = 0;
        g->steps->teams_bytes = 0;
        if (alloc_refused() || hipMalloc((void **)&t.block, (size_t)need) != hipSuccess) {
            t.block = nullptr;
            return set_error(MG_ERR_OOM, "batched search state of %lld bytes: allocation failed", (long long)need);
        }
        t.cap = need;
        g->steps->teams_bytes = need;
    }
    TeamsArgs a{};
    a.ctl = reinterpret_cast<TeamsCtl *>(t.block + at_ctl);
    a.team = reinterpret_cast<TeamCtl *>(t.block + at_team);
    a.recs = reinterpret_cast<uint64_t *>(t.block + at_recs);
    a.bits = reinterpret_cast<uint32_t *>(t.block + at_bits);
    int *const own = reinterpret_cast<int *>(t.block + at_rows), *const d_pairs = reinterpret_cast<int *>(t.block + at_pairs);
    a.rows = direct ? out : own;
    a.row_start = d_pairs;
    a.srcs = d_pairs + MG_BATCH_MAX + 1;
    // (the graph's pinned control block is free between searches)
    static_assert(sizeof(TeamsCtl) <= sizeof(Ctl), "copied to the pinned block");
    TeamsCtl *const h = reinterpret_cast<TeamsCtl *>(g->ws.h_ctl);
    a.off = g->row_off;
    a.adj = g->col;
    a.w = g->w;
    a.n = g->n;
    a.nwords = nwords;
    a.k = k;
    a.per_xcd = per_xcd;
    a.wgs = std::min(TEAM_WGS, TEAMS_GRID / teams);
    a.limit = o.iter_num;
    // bucket width as mg_sssp's narrow levels: four largest weights
    a.delta = o.sssp_delta < 0 ? LLONG_MAX / 4 : o.sssp_delta > 0 ? o.sssp_delta : std::max<long long>(1, 4LL * g->max_weight);
    const int unreached = sssp ? INT_MAX : -1;
    MG_HIP(hipEventRecord(g->ev0, g->stream));
    MG_HIP(hipMemcpyAsync(d_pairs, pairs.data(), 4 * pairs.size(), hipMemcpyHostToDevice, g->stream));
    hipLaunchKernelGGL(teams_init, dim3(grid_blocks_cap(std::max<int64_t>(cells / 4, 4LL * teams * nwords), BLK, 4 * MAX_GRID)),
                       dim3(BLK), 0, g->stream, a, unreached);
    const int grid = teams * teams_launch(a.wgs);
    if (sssp) hipLaunchKernelGGL(teams_sssp, dim3(grid), dim3(BLK), 0, g->stream, a);
    else hipLaunchKernelGGL(teams_bfs, dim3(grid), dim3(BLK), 0, g->stream, a);
    if (stats)
        hipLaunchKernelGGL(teams_stats, dim3(std::max(1, std::min(64, grid_blocks(g->n, BLK))), k), dim3(BLK), 0,
                           g->stream, a, unreached);
    MG_HIP(hipGetLastError());
    MG_HIP(hipEventRecord(g->ev1, g->stream));
    MG_HIP(hipMemcpyAsync(h, a.ctl, sizeof(TeamsCtl), hipMemcpyDeviceToHost, g->stream));
    MG_HIP(hipStreamSynchronize(g->stream));
    *wgs = a.wgs;
    *end = h->end;
    if (*end != TEAMS_DONE) return MG_OK;
    float ms = 0;
    MG_HIP(hipEventElapsedTime(&ms, g->ev0, g->ev1));
    if (stats) {
        std::memset(stats, 0, sizeof *stats);
        stats->iterations = h->levels;
        stats->edges_examined = (int64_t)h->edges;
        stats->edges_traversed = (int64_t)h->te;
        stats->vertices_reached = (int64_t)h->nr;
        stats->device_ms = ms;
    }
    if (!direct)
        if (const int rc = deliver(g, out, own, 4 * (size_t)cells, o.out_on_device)) return rc;
    if (stats) stats->host_ms = timer.ms();
    return MG_OK;
}

int teams_try(mg_graph *g, bool sssp, const int32_t *row_of, const int32_t *srcs, int32_t npairs, int32_t k, int32_t *out,
              const mg_options &o, mg_stats *stats, const CallTimer &timer, bool *done) {
    *done = false;
    TeamsRule &rule = g->steps->teams_rule[sssp];
    if (g->m >= TEAMS_DEGREE * (int64_t)g->n || !rule.wanted()) return MG_OK;
    for (bool again = false;;) {
        int end = TEAMS_DONE, wgs = 0;
        const int rc = teams_batch(g, sssp, row_of, srcs, npairs, k, out, o, stats, timer, &end, &wgs);
        if (route_refused(rc)) break;
        if (rc || end == TEAMS_DONE) {
            *done = true;
            if (!rc) rule.succeeded();
            return rc;
        }
        if (!rule.retry(end, wgs, TEAM_WGS, again)) {
            if (rule.skip > 0 && g->steps->teams_bytes > TEAMS_KEEP) teams_release(g);  // (else the next call tries again)
            return MG_OK;
        }
        again = again || end == TEAMS_SHORT;
    }
    teams_release(g);  // room for the general route
    return MG_OK;
}

}  // namespace mg
