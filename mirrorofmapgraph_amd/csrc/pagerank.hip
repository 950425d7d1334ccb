// PageRank: the engine's specialised path for the pagerank program
// (Algorithms/PageRank/PageRank.h).
//
// The reference program gathers over in-edges (GATHER_IN_EDGES, PageRank.h:197-200)
// the value rank[u] / outdeg[u] (gather_edge, :233-243), sums it (gather_sum), and
// applies new = 0.15f + (1.0f - 0.15f) * sum, marking the vertex changed when
// |old - new| >= 0.01f (apply, :257-283); the next frontier is the out-neighbours
// of changed vertices (expand_edge, :355-362), deduplicated.  Gathers of one
// iteration all read the previous ranks (the enactor runs gather before apply),
// i.e. frontier-restricted Jacobi.  The enactor materialises (dst, value) pairs
// per in-edge and reduces them with a segmented reduction (enactor:1503-1596).
//
// Here the gather is a pull over the in-edge view that fuses gather, apply and the
// frontier test: a vertex is active at iteration i > 0 exactly when one of its
// in-neighbours changed at iteration i-1 (that is the reference's expand), so one
// pass per iteration reads each in-edge once, sums precomputed contributions
// contrib[u] = rank[u] / (float)outdeg[u] (the same float division as gather_edge),
// and applies.  Summation order is fixed, so results are deterministic:
//   in-degree <= PR_T1   one lane, sequentially in in-edge order (the wave gathers the
//                        edges of a run of such vertices together, into LDS);
//   up to a piece        one wave: lane l sums edges l, l+64, ... in order, then an
//                        xor-butterfly over offsets 32,16,8,4,2,1;
//   longer               pieces summed as above, then their sums added in order.
// MG_PR_ALL updates every vertex each iteration (all-vertex Jacobi) and can stop on
// the L1 change, reduced in a fixed order as well.
//
// An iteration is one launch: the wave that finishes a high in-degree vertex's last chunk
// adds its chunk sums, and the workgroup that finishes last closes the iteration
// (counters in device memory, what they guard stored and loaded device-coherently).
//
// Bound: the gathers contrib[u], an L2 request for each distinct line of a wave's 64.  On
// graphs whose hubs have the lowest ids (the degree-ordered twin; R-MAT as generated) every
// workgroup copies the first PR_HUBS contributions into LDS, and a gather below PR_HUBS is
// an LDS read: 50% of the edges of the directed R-MAT scale 21 (33.5M edges), 57% at scale
// 20.  60 KB let two workgroups share a CU: 32768 contributions in 128 KB, one workgroup a
// CU, took 136 us an iteration where 16384 and two took 130.  Gathering a low in-degree
// vertex in a lane of its own made 64 lanes read 64 lists; a wave that gathers a run of them
// in edge order reads adjacency lines once (130 -> 115).
// Measured, us an iteration, directed R-MAT, edge factor 16, degree-ordered (as generated):
//   scale 16   28 -> 15 (28 -> 14)
//   scale 19   57 -> 33 (79 -> 45)
//   scale 21   158 -> 112 (233 -> 179)
// of which at scale 21 7.5 are the launch, the copy and the close, 55 with the adjacency read
// and the sums made but no contribution loaded.  Without LDS hubs 147.
#include <vector>

#include "frontier.h"

namespace mg {

// In-degrees a lane sums alone: 32, 48, 64 and 128 took 129, 115, 115 and 120 us at scale 21,
// 48 and 64 39 and 42 at scale 19.
constexpr int PR_T1 = 48;
constexpr int PR_BLK = 1024;        // threads of pr_iterate
constexpr int PR_HUBS = 15360;      // contributions kept in LDS: 60 KB, two workgroups a CU
constexpr int PR_BUF = 256;         // edges of a run in LDS at a time (per wave)
// A wave's piece of work (a run of low in-degree vertices, or a part of a list) has
// m / PR_PIECES edges, so that small graphs have pieces for all 8192 waves and large ones few
// records: at 1024 edges whatever the size scales 16 and 19 took 20 and 34 us, now 15 and 33;
// least pieces of 128 took 17 at scale 16.
constexpr int PR_PIECES = 16384;
constexpr int PR_PIECE_MIN = 256, PR_PIECE_MAX = 2048;
// One edge in so many has to come from a hub for the copy to pay: it costs 1 us and the LDS
// reads of every gather, a gather saved 1/230000 us.
constexpr int PR_HUB_SHARE = 5;

struct PrArgs {
    Ctl *ctl;
    const int *in_off, *in_adj, *row_off;
    float *rank;
    float *contrib[2];
    uint32_t *chg[3];
    const ChunkRec *runs;    // {first vertex, -, -, vertices}
    const ChunkRec *lists;   // chunks (pad: the vertex's index in bigv), then medium lists (pad -1)
    const int *bigv;
    float *part;
    int *pact;
    int *left;               // per high in-degree vertex: chunks summed; then workgroups finished
    double *partials;        // per workgroup: L1 change, changed vertices
    int n, nwords, nruns, nlists, nbig, G;
    int mode;
    float base, damp, eps;
    double tol_n;
};

struct PrIter {
    int it;
    const float *c_old;
    float *c_new;
    const uint32_t *prev;
    uint32_t *cur;
};

__device__ __forceinline__ PrIter pr_iter(const PrArgs &a) {
    PrIter s;
    s.it = a.ctl->level;
    s.c_old = a.contrib[s.it & 1];
    s.c_new = a.contrib[(s.it + 1) & 1];
    s.prev = a.chg[(s.it + 2) % 3];
    s.cur = a.chg[s.it % 3];
    return s;
}

// Applies the gathered sum s to v; returns |new - old| (0 when inactive).  ranks: the rank
// itself is read and stored (iterations whose ranks nothing looks at need only the
// contributions).
__device__ __forceinline__ double pr_apply(const PrArgs &a, const PrIter &I, int v, int od, float s, bool active,
                                           bool ranks, int &nchanged) {
    if (!active) {
        I.c_new[v] = I.c_old[v];
        return 0.0;
    }
    const float nv = a.base + a.damp * s;
    I.c_new[v] = nv / (float)od;
    if (!ranks) return 0.0;
    const float old = a.rank[v];
    a.rank[v] = nv;
    if (a.mode == MG_PR_GAS && !(fabsf(old - nv) < a.eps)) {
        atomicOr(&I.cur[v >> 5], 1u << (v & 31));
        if (od > 0) ++nchanged;  // only vertices with out-edges put anything in the next frontier
    }
    return fabs((double)nv - (double)old);
}

__global__ void pr_init(PrArgs a, int iter_limit) {
    for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < a.n; v += gridDim.x * blockDim.x) {
        a.rank[v] = a.base;
        a.contrib[0][v] = a.base / (float)(a.row_off[v + 1] - a.row_off[v]);
        a.contrib[1][v] = a.contrib[0][v];
    }
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < a.nwords; i += gridDim.x * blockDim.x) {
        a.chg[0][i] = 0;
        a.chg[1][i] = 0;
        a.chg[2][i] = 0;
    }
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < a.nbig + LAST_WG_INTS; i += gridDim.x * blockDim.x) a.left[i] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl_reset(a.ctl, a.n, iter_limit, a.n);
}

// contrib[u]: from LDS below the hub count h, else from memory (lanes with a hub read one
// shared entry there, so no branch waits between the loads of a batch).
template <bool HUB>
struct PrGather {
    const float *c_old, *hubs;
    int h, other;  // other: an entry of c_old for the lanes that have theirs in LDS
    template <int K>
    __device__ __forceinline__ void get(const int (&u)[K], float (&out)[K]) const {
        if (!HUB) {
#pragma unroll
            for (int j = 0; j < K; ++j) out[j] = c_old[u[j]];
            return;
        }
        float g[K];
#pragma unroll
        for (int j = 0; j < K; ++j) g[j] = c_old[u[j] < h ? other : u[j]];
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const float l = hubs[u[j] < h ? u[j] : 0];
            out[j] = u[j] < h ? l : g[j];
        }
    }
};

// Wave sum of edges [beg, end): lane-strided, then xor-butterfly.  `act` is OR-ed
// over the wave as well.
template <bool HUB>
__device__ __forceinline__ float wave_gather(const PrArgs &a, const PrIter &I, const PrGather<HUB> &c, int beg, int end,
                                             bool &act) {
    const int lane = lane_id();
    const bool all = act;  // activity already known: skip the bitmap
    float s = 0.0f;
    bool any = false;
    // lane l sums edges l, l+64, ... in order, eight then four in flight (full groups load
    // unconditionally), then the remainder one at a time
    int e = beg + lane;
    auto batch = [&](auto kc) {
        constexpr int K = decltype(kc)::value;
        for (; e + (K - 1) * WAVE < end; e += K * WAVE) {
            int u[K];
            float cv[K];
#pragma unroll
            for (int j = 0; j < K; ++j) u[j] = a.in_adj[e + j * WAVE];
            c.get(u, cv);
            if (!all) {
#pragma unroll
                for (int j = 0; j < K; ++j) any = any || test_bit(I.prev, u[j]);
            }
#pragma unroll
            for (int j = 0; j < K; ++j) s = s + cv[j];
        }
    };
    batch(std::integral_constant<int, 8>());
    batch(std::integral_constant<int, 4>());
    batch(std::integral_constant<int, 1>());
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s = s + __shfl_xor(s, o);
    act = act || (wave_ballot(any) != 0);
    return s;
}

// One iteration.
template <bool HUB>
__global__ __launch_bounds__(PR_BLK, 8) void pr_iterate(PrArgs a) {
    Ctl *c = a.ctl;
    if (c->done) return;
    __shared__ float s_hubs[HUB ? PR_HUBS : 1];
    __shared__ float s_buf[PR_BLK / WAVE][PR_BUF];
    const PrIter I = pr_iter(a);
    const bool all = a.mode == MG_PR_ALL || I.it == 0;
    const bool ranks = a.mode != MG_PR_ALL || a.tol_n > 0 || I.it + 1 >= c->iter_limit;
    const int tid = blockIdx.x * PR_BLK + (int)threadIdx.x, nt = gridDim.x * PR_BLK;
    PrGather<HUB> cg{I.c_old, s_hubs, 0, 0};
    if (HUB) {
        const int h = min(a.n, PR_HUBS);
        const float4 *src = reinterpret_cast<const float4 *>(I.c_old);
        for (int i = threadIdx.x; i < h / 4; i += PR_BLK) reinterpret_cast<float4 *>(s_hubs)[i] = src[i];
        if ((int)threadIdx.x < h % 4) s_hubs[h / 4 * 4 + threadIdx.x] = I.c_old[h / 4 * 4 + threadIdx.x];
        cg.h = h;
        cg.other = min(h, a.n - 1);
        __syncthreads();
    }
    // the bitmap filled at iteration it+1 is cleared now
    uint32_t *clr = a.chg[(I.it + 1) % 3];
    for (int i = tid; i < a.nwords; i += nt) clr[i] = 0;
    double delta = 0;
    int nchanged = 0;
    // chunks of high in-degree vertices and medium vertices, a wave each; the next record is
    // loaded, and the out-degree on its way, while a list is summed
    const int lane = lane_id(), nw = nt / WAVE;
    ChunkRec r{};
    if (tid / WAVE < a.nlists) r = a.lists[tid / WAVE];
    for (int t = tid / WAVE; t < a.nlists; t += nw) {
        const ChunkRec next = a.lists[min(t + nw, a.nlists - 1)];
        const int v = r.v, big = r.pad;
        const int od = a.row_off[v + 1] - a.row_off[v];
        bool act = all;
        const float s = wave_gather<HUB>(a, I, cg, r.beg, r.end, act);
        r = next;
        if (big < 0) {
            if (lane == 0) delta += pr_apply(a, I, v, od, s, act, ranks, nchanged);
            continue;
        }
        const int c0 = a.bigv[big], c1 = a.bigv[big + 1];
        int old = 0;
        if (lane == 0) {
            __hip_atomic_store(&a.part[t], s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&a.pact[t], (int)act, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // stored before it is counted
            old = atomicAdd(&a.left[big], 1);
        }
        if (__builtin_amdgcn_readfirstlane(old) != c1 - c0 - 1) continue;
        // the vertex's last chunk: its sums in chunk order, 64 loaded together
        float sum = 0.0f;
        bool hot = all;
        for (int ci = c0; ci < c1; ci += WAVE) {
            const int i = min(ci + lane, c1 - 1);
            const float p = __hip_atomic_load(&a.part[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const int q = ld_dev(&a.pact[i]);
            hot = hot || wave_ballot(ci + lane < c1 && q != 0) != 0;
            const int m = min(WAVE, c1 - ci);
            for (int j = 0; j < m; ++j) {
                const float x = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, p), j));
                sum = ci == c0 && j == 0 ? x : sum + x;
            }
        }
        if (lane == 0) {
            a.left[big] = 0;
            delta += pr_apply(a, I, v, od, sum, hot, ranks, nchanged);
        }
    }
    // low in-degree vertices: a wave gathers the edges of a run, each lane adds its vertex's
    float *buf = s_buf[threadIdx.x / WAVE];
    if (tid / WAVE < a.nruns) r = a.runs[tid / WAVE];
    for (int t = tid / WAVE; t < a.nruns; t += nw) {
        const ChunkRec next = a.runs[min(t + nw, a.nruns - 1)];
        const bool mine = lane < r.pad;
        const int w = mine ? r.v + lane : r.v;
        const int od = a.row_off[w + 1] - a.row_off[w];
        const int beg = a.in_off[r.v + min(lane, r.pad)], end = a.in_off[r.v + min(lane + 1, r.pad)];
        const int e0 = __builtin_amdgcn_readfirstlane(beg), e1 = a.in_off[r.v + r.pad];
        float s = 0.0f;
        bool act = all;
        for (int p0 = e0; p0 < e1; p0 += PR_BUF) {
            constexpr int K = PR_BUF / WAVE;
            int u[K];
            float cv[K];
#pragma unroll
            for (int j = 0; j < K; ++j) u[j] = a.in_adj[min(p0 + j * WAVE + lane, e1 - 1)];
            cg.get(u, cv);
#pragma unroll
            for (int j = 0; j < K; ++j) buf[j * WAVE + lane] = cv[j];
            if (!all) {
#pragma unroll
                for (int j = 0; j < K; ++j) {
                    const uint64_t m = wave_ballot(test_bit(I.prev, u[j]));
                    const int lo = max(beg - p0 - j * WAVE, 0), hi = min(end - p0 - j * WAVE, WAVE);
                    if (hi > lo) act = act || ((m >> lo) & (~0ull >> (WAVE - (hi - lo)))) != 0;
                }
            }
            wave_sync();
            for (int e = max(beg, p0); e < min(end, p0 + PR_BUF); ++e) s = s + buf[e - p0];
            wave_sync();  // the next edges overwrite these
        }
        if (mine) delta += pr_apply(a, I, w, od, s, act, ranks, nchanged);
        r = next;
    }
    // the last workgroup closes the iteration, adding the workgroups' sums in order
    if (ranks) {
        delta = block_sum<PR_BLK>(delta);
        const long long nch = block_sum<PR_BLK>((long long)nchanged);
        if (threadIdx.x == 0) {
            __hip_atomic_store(&a.partials[2 * blockIdx.x], delta, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&a.partials[2 * blockIdx.x + 1], (double)nch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
    }
    if (!last_workgroup(a.left + a.nbig)) return;
    double l1 = 0, changed = 0;
    if (ranks) {
        for (int i = threadIdx.x; i < (int)gridDim.x; i += PR_BLK) {
            l1 += __hip_atomic_load(&a.partials[2 * i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            changed += __hip_atomic_load(&a.partials[2 * i + 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        l1 = block_sum<PR_BLK>(l1);
        changed = block_sum<PR_BLK>(changed);
    }
    if (threadIdx.x == 0) {
        c->dsum = l1;
        c->level = I.it + 1;
        c->changed = (int)changed;
        bool done = I.it + 1 >= c->iter_limit;
        if (a.mode == MG_PR_GAS && changed == 0) done = true;
        if (a.mode == MG_PR_ALL && a.tol_n > 0 && l1 < a.tol_n) done = true;
        c->done = done;
    }
}

// Edges whose source id is below `lim`.
__global__ __launch_bounds__(BLK) void pr_count_below(const int *adj, int64_t m, int lim, unsigned long long *out) {
    long long k = 0;
    for (int64_t e = blockIdx.x * (int64_t)BLK + threadIdx.x; e < m; e += (int64_t)gridDim.x * BLK) k += adj[e] < lim;
    k = block_sum<BLK>(k);
    if (threadIdx.x == 0 && k) atomicAdd(out, (unsigned long long)k);
}

// Builds (once per graph and in-edge view) the records of the runs and lists, on the host from the in-edge offsets.
static int pr_buckets(mg_graph *g, const int *d_in_off, const int *d_in_adj) {
    Workspace &ws = g->ws;
    if (ws.pr_view == d_in_off) return MG_OK;
    const int n = g->n;
    std::vector<int32_t> off((size_t)n + 1);
    MG_HIP(copy_on(g->stream, off.data(), d_in_off, 4 * ((size_t)n + 1), hipMemcpyDeviceToHost));
    const int piece = (int)std::clamp<int64_t>(g->m / PR_PIECES / WAVE * WAVE, PR_PIECE_MIN, PR_PIECE_MAX);
    std::vector<int32_t> bigv;
    std::vector<ChunkRec> mid, ch, runs;
    for (int v = 0; v < n; ++v) {
        const int d = off[v + 1] - off[v];
        if (d <= PR_T1) {
            if (!runs.empty() && runs.back().v + runs.back().pad == v && runs.back().pad < WAVE &&
                off[v + 1] - off[runs.back().v] <= piece)
                runs.back().pad++;
            else
                runs.push_back(ChunkRec{v, 0, 0, 1});
            continue;
        }
        if (d <= piece) {
            mid.push_back(ChunkRec{v, off[v], off[v + 1], -1});
        } else {
            bigv.push_back((int)ch.size());
            for (int b = off[v]; b < off[v + 1]; b += piece) ch.push_back(ChunkRec{v, b, std::min(b + piece, off[v + 1]), (int)bigv.size() - 1});
        }
    }
    bigv.push_back((int)ch.size());
    free_dev(ws.pr_lists);
    free_dev(ws.pr_bigv);
    free_dev(ws.pr_part);
    free_dev(ws.pr_pact);
    free_dev(ws.pr_left);
    free_dev(ws.pr_runs);
    ws.pr_left = nullptr;
    ws.pr_runs = nullptr;
    ws.pr_lists = nullptr;
    ws.pr_bigv = nullptr;
    ws.pr_part = nullptr;
    ws.pr_pact = nullptr;
    ws.pr_view = nullptr;
    int rc;
    const size_t nchunks = ch.size();
    ch.insert(ch.end(), mid.begin(), mid.end());
    if ((rc = alloc_chunks(&ws.pr_lists, ch.size())) || (rc = alloc_i32(&ws.pr_bigv, bigv.size())) ||
        (rc = alloc_f32(&ws.pr_part, nchunks)) || (rc = alloc_i32(&ws.pr_pact, nchunks)) ||
        (rc = alloc_i32(&ws.pr_left, bigv.size() + LAST_WG_INTS)) || (rc = alloc_chunks(&ws.pr_runs, runs.size())))
        return rc;
    // the share of the edges whose source is among the first PR_HUBS ids
    MG_HIP(hipMemsetAsync(ws.d_reach, 0, 16, g->stream));
    hipLaunchKernelGGL(pr_count_below, dim3(grid_blocks(g->m, BLK)), dim3(BLK), 0, g->stream, d_in_adj, g->m, PR_HUBS,
                       ws.d_reach);
    MG_HIP(hipGetLastError());
    MG_HIP(copy_on(g->stream, ws.h_reach, ws.d_reach, 8, hipMemcpyDeviceToHost));
    ws.pr_hubs = (int64_t)ws.h_reach[0] * PR_HUB_SHARE >= g->m;
    if (!ch.empty()) MG_HIP(copy_on(g->stream, ws.pr_lists, ch.data(), sizeof(ChunkRec) * ch.size(), hipMemcpyHostToDevice));
    MG_HIP(copy_on(g->stream, ws.pr_bigv, bigv.data(), 4 * bigv.size(), hipMemcpyHostToDevice));
    if (!runs.empty())
        MG_HIP(copy_on(g->stream, ws.pr_runs, runs.data(), sizeof(ChunkRec) * runs.size(), hipMemcpyHostToDevice));
    ws.pr_nruns = (int)runs.size();
    ws.pr_nlists = (int)ch.size();
    ws.pr_nbig = (int)bigv.size() - 1;
    ws.pr_view = d_in_off;
    return MG_OK;
}

}  // namespace mg

using namespace mg;

extern "C" int mg_pagerank(mg_graph *g, float *rank_out, const mg_options *opt, mg_stats *stats) {
    CallTimer timer;
    mg_options o;
    int rc = begin_search(g, opt, &o);
    if (rc) return rc;
    std::lock_guard<std::mutex> lock(g->mu);
    if (o.pr_mode != MG_PR_GAS && o.pr_mode != MG_PR_ALL)
        return set_error(MG_ERR_INVALID_ARG, "mg_pagerank: unknown pr_mode %d", o.pr_mode);
    const bool sym = g->flags & MG_GRAPH_SYMMETRIC;
    if (!sym && !g->col_off)
        return set_error(MG_ERR_UNSUPPORTED, "mg_pagerank: needs the in-edge view (MG_GRAPH_BUILD_CSC) or a symmetric graph");
    if (o.directed == 0 && !sym)
        return set_error(MG_ERR_UNSUPPORTED, "mg_pagerank: directed=0 is supported on symmetric graphs only");
    if (o.engine == MG_ENGINE_GAS) {
        if (o.pr_mode != MG_PR_GAS || o.pr_teleport != 0.15f || o.pr_active_eps != 0.01f)
            return set_error(MG_ERR_UNSUPPORTED, "MG_ENGINE_GAS runs the reference pagerank program (pr_mode "
                                                 "MG_PR_GAS, teleport 0.15, eps 0.01)");
        return gas_pagerank(g, rank_out, o, stats, timer);
    }
    g = search_graph(g, o, nullptr);  // the degree-ordered twin, when the graph keeps one
    if ((rc = ensure_workspace(g)) || (rc = ensure_pr_workspace(g))) return rc;
    const int *in_off = sym ? g->row_off : g->col_off;
    const int *in_adj = sym ? g->col : g->row_idx;
    if ((rc = pr_buckets(g, in_off, in_adj))) return rc;
    Workspace &ws = g->ws;
    PrArgs a{};
    a.ctl = ws.ctl;
    a.in_off = in_off;
    a.in_adj = in_adj;
    a.row_off = g->row_off;
    a.rank = ws.rank;
    a.contrib[0] = ws.contrib[0];
    a.contrib[1] = ws.contrib[1];
    for (int i = 0; i < 3; ++i) a.chg[i] = ws.bm[i];
    a.lists = ws.pr_lists;
    a.runs = ws.pr_runs;
    a.nruns = ws.pr_nruns;
    a.bigv = ws.pr_bigv;
    a.part = ws.pr_part;
    a.pact = ws.pr_pact;
    a.left = ws.pr_left;
    a.partials = ws.partials;
    a.n = g->n;
    a.nwords = ws.nwords;
    a.nlists = ws.pr_nlists;
    a.nbig = ws.pr_nbig;
    a.mode = o.pr_mode;
    a.base = o.pr_teleport;
    a.damp = 1.0f - o.pr_teleport;
    a.eps = o.pr_active_eps;
    a.tol_n = (double)o.pr_tol * (double)g->n;
    // two workgroups a CU; fewer on small graphs
    const bool hubs = ws.pr_hubs;
    a.G = grid_blocks_cap(std::max<int64_t>(a.nruns, a.nlists) * WAVE, PR_BLK, 512);

    MG_HIP(hipEventRecord(g->ev0, g->stream));
    hipLaunchKernelGGL(pr_init, dim3(grid_blocks(g->n, BLK)), dim3(BLK), 0, g->stream, a, o.iter_num);
    MG_HIP(hipGetLastError());
    auto step = [&]() -> int {
        if (hubs) hipLaunchKernelGGL(pr_iterate<true>, dim3(a.G), dim3(PR_BLK), 0, g->stream, a);
        else hipLaunchKernelGGL(pr_iterate<false>, dim3(a.G), dim3(PR_BLK), 0, g->stream, a);
        MG_HIP(hipGetLastError());
        return MG_OK;
    };
    // the captured steps bake in the per-call constants: key on all of them
    uint64_t key = (uint64_t)a.mode;
    for (uint64_t x : {(uint64_t)__builtin_bit_cast(uint32_t, a.base), (uint64_t)__builtin_bit_cast(uint32_t, a.eps),
                       (uint64_t)__builtin_bit_cast(uint64_t, a.tol_n), (uint64_t)(uintptr_t)in_off})
        key = mix64(key ^ x);
    if ((rc = drive(g, step, (int64_t)std::max(o.iter_num, 0) + 1, KIND_PR, key))) return rc;
    rc = finish_search(g, stats, nullptr, 0, ws.rank, 4 * (size_t)g->n,
                       plan_delivery(g, rank_out, 4 * (size_t)g->n, o.out_on_device), timer);
    if (rc) return rc;
    if (stats) {
        stats->edges_traversed = g->m * (int64_t)stats->iterations;
        stats->vertices_reached = g->n;
    }
    return MG_OK;
}
