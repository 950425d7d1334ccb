// Batched BFS that keeps every level's frontier: the path of mg_bfs_batch on graphs whose
// searches are shallow.
//
// batch.hip writes a depth row entry for each (vertex, source) pair as the pair is
// reached: 4-byte stores scattered over 256 rows, on a row array cleared first, and on a
// degree-ordered twin every row gathered back afterwards.  Here level l's frontier masks
// stay in H[l] (n masks of 256 bits, the slots' rows buffer holds LEVELS_MAX of them) and
// one pass at the end (bl_expand) turns the levels of each vertex into depths, row by row
// in the caller's order, straight into the result.  What that takes away from a level:
//   * no depth stores and no finalize pass: the next frontier is H[L + 1] itself, and the
//     visited masks lag one level (visited before level L + 1 = V | H[L]; whoever handles
//     a frontier vertex folds H[L] into V);
//   * no copy of the masks: push ORs into H[L + 1] (cleared two levels ahead), pull stores
//     it.
// A search deeper than LEVELS_MAX - 2 levels stops and is run again by batch.hip, as are
// all later ones on the graph.
//
// Measured (R-MAT scale 20 with its twin, m = 31 M, 256 sources, result in device memory):
// 6.4 -> 1.28 ms a call.  The levels take 0.8 ms, bound by the pulls' random 32-byte mask
// gathers; bl_expand 0.31 ms for 1 GB of rows (3.4 TB/s; the copy kernel moves 5.2).
// Pushing the second level (frontier out-edges just under m / 4) took 0.98 ms where
// pulling it takes 0.34, hence LEVELS_ALPHA = 16 as the default switch.
#include "batch.h"

namespace mg {

constexpr int LEVELS_MAX = 32;  // levels the rows buffer holds: 256 slots x 4 bytes = 32 masks of 32 bytes
static_assert(MG_BATCH_MAX * 4 == LEVELS_MAX * 32, "the rows of a full context hold the levels");
// Pull: a vertex whose first BU_INLINE in-edges leave a source open goes to a wave; what
// is left of a longer list is cut into pieces of LEVELS_PIECE edges, a wave each (one wave
// walked a hub's 100K edges alone: 567 us of a 680 us level).
constexpr int LEVELS_PIECE = 1024;
constexpr int LEVELS_DEEP = 1 << 29;  // Ctl::changed: the search outgrew the levels

struct LevelsArgs {
    Ctl *ctl;
    SlotCtl *sc;
    const int *off, *adj;        // push view (CSR)
    const int *in_off, *in_adj;  // pull view (in-edges), nullptr when none
    uint4 *V, *H;                // visited masks (one level behind); LEVELS_MAX x n frontier masks
    uint32_t *act[2];            // active-vertex bitmaps
    int *hard;                   // pull: vertices handed to a wave
    ChunkRec *tasks;
    int64_t task_cap;
    FrontierArgs fa;             // level counters only (part)
    int n, nwords, G;
    __device__ uint4 *level(int l) const { return H + 2 * (int64_t)l * n; }
};

__device__ __forceinline__ M8 none8() { return M8{make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0)}; }

__global__ void bl_init(LevelsArgs a, int iter_limit, int can_pull, int alpha, int beta, long long m) {
    const int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, nt = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = tid; i < 2 * (int64_t)a.n; i += nt) a.V[i] = make_uint4(0, 0, 0, 0);
    for (int64_t i = tid; i < 4 * (int64_t)a.n; i += nt) a.H[i] = make_uint4(0, 0, 0, 0);  // levels 0 and 1
    for (int64_t i = tid; i < a.nwords; i += nt) {
        a.act[0][i] = 0;
        a.act[1][i] = 0;
    }
    int *sci = reinterpret_cast<int *>(a.sc);
    for (int64_t i = tid; i < (int64_t)(sizeof(SlotCtl) / 4); i += nt) sci[i] = 0;
    if (blockIdx.x != 0) return;
    clear_parts(a.fa);
    if (threadIdx.x != 0) return;
    Ctl *c = a.ctl;
    ctl_reset(c, a.n, iter_limit, 1);
    c->can_bu = can_pull;
    c->m_unexplored = m;  // pull once the frontier's out-edges exceed m / alpha
    c->alpha = alpha;
    c->beta = beta;
}

// One thread per (slot, source) pair.
__global__ void bl_seed(LevelsArgs a, SeedList sl) {
    const int i = threadIdx.x;
    if (i >= sl.n) return;
    const int s = sl.slot[i], v = sl.src[i];
    atomicOr(reinterpret_cast<uint32_t *>(a.H + 2 * (int64_t)v) + (s >> 5), 1u << (s & 31));
    atomicOr(&a.act[0][v >> 5], 1u << (v & 31));
    atomicOr(&a.sc->assigned[s >> 5], 1u << (s & 31));
}

// One workgroup: closes the pending level.
__global__ __launch_bounds__(SMALL_BLK) void bl_close(LevelsArgs a) {
    Ctl *c = a.ctl;
    if (c->done) return;
    if (threadIdx.x == 0) c->steps++;
    if (!c->pending) return;
    long long nf, mf, ex;
    take_level_parts<SMALL_BLK>(a.fa, nf, mf, ex);
    if (threadIdx.x != 0) return;
    const int L = c->level;
    int dir = c->dir;
    if (dir == DIR_BU) c->bu_levels++;
    if (c->can_bu) {
        if (dir == DIR_TD && mf * c->alpha > c->m_unexplored) dir = DIR_BU;
        else if (dir == DIR_BU && mf * c->beta < c->m_unexplored) dir = DIR_TD;
    }
    c->dir = dir;
    c->pending = 0;
    c->nchunks = 0;
    c->nhard = 0;
    c->level = L + 1;
    c->nf_prev = (int)nf;
    if (nf == 0 || L + 1 >= c->iter_limit) {
        c->done = 1;
    } else if (L + 2 >= LEVELS_MAX) {
        c->changed |= LEVELS_DEEP;
        c->done = 1;
    }
}

// v's frontier bits that u has not seen yet go to u's next mask; u's first bit of the level
// marks and counts it.
__device__ __forceinline__ void bl_push(const LevelsArgs &a, const M8 &fv, int u, const uint4 *cur, uint4 *next,
                                        uint32_t *act_next, long long &nf, long long &mf) {
    const M8 nw = andnot8(andnot8(fv, ld8(a.V, u)), ld8(cur, u));
    if (!any8(nw)) return;
    uint32_t *nu = reinterpret_cast<uint32_t *>(next + 2 * (int64_t)u);
#pragma unroll
    for (int w = 0; w < 8; ++w) {
        const uint32_t b = word8(nw, w);
        if (b) atomicOr(&nu[w], b);
    }
    if (!test_bit(act_next, u) && set_bit_first(act_next, u)) {
        ++nf;
        mf += a.off[u + 1] - a.off[u];
    }
}

__global__ __launch_bounds__(BLK) void bl_a(LevelsArgs a) {
    Ctl *c = a.ctl;
    if (c->done) return;
    const int L = c->level;
    const uint4 *cur = a.level(L);
    uint4 *next = a.level(L + 1);
    uint32_t *act_next = a.act[(L + 1) & 1];
    long long nf = 0, mf = 0;
    // the level after the next starts empty (level L + 1 was cleared during level L - 1)
    if (L + 2 < LEVELS_MAX) {
        uint4 *z = a.level(L + 2);
        for (int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x; i < 2 * (int64_t)a.n; i += (int64_t)gridDim.x * BLK)
            z[i] = make_uint4(0, 0, 0, 0);
    }
    if (c->dir == DIR_TD) {
        __shared__ int s_w[BLK / WAVE];
        __shared__ int s_tb;
        for_each_bit_clear(a.act[L & 1], a.nwords, [&](int v) {
            int beg = 0, deg = 0;
            M8 fv = none8();
            if (v >= 0) {
                beg = a.off[v];
                deg = a.off[v + 1] - beg;
                fv = ld8(cur, v);
                st8(a.V, v, or8(ld8(a.V, v), fv));
            }
            const int nt = deg > LANE_T ? (deg + TASK - 1) / TASK : 0;
            int tot;
            const int tex = block_exclusive_scan<BLK>(nt, s_w, &tot);
            if (tot > 0) {
                if (threadIdx.x == 0) s_tb = atomicAdd(&c->nchunks, tot);
                __syncthreads();
                for (int t = 0; t < nt; ++t) {
                    const int64_t slot = (int64_t)s_tb + tex + t;
                    if (slot < a.task_cap)
                        a.tasks[slot] = ChunkRec{v, beg + t * TASK, min(beg + (t + 1) * TASK, beg + deg), 0};
                    else
                        atomicOr(&c->changed, 1 << 30);
                }
                __syncthreads();
            }
            if (nt == 0 && deg > 0)
                for (int e = beg; e < beg + deg; ++e) bl_push(a, fv, a.adj[e], cur, next, act_next, nf, mf);
        });
    } else {
        __shared__ int s_w[BLK / WAVE];
        __shared__ int s_hb;
        const int lane = lane_id();
        const M8 full = ld8(reinterpret_cast<const uint4 *>(a.sc->assigned), 0);
        uint32_t *act_cur = a.act[L & 1];
        for (int base = blockIdx.x * BLK; base < a.n; base += gridDim.x * BLK) {
            const int u = base + (int)threadIdx.x;
            bool found = false, hard = false;
            int pieces = 0;
            if (u < a.n) {
                const M8 own = ld8(cur, u);
                M8 vu = ld8(a.V, u);
                if (any8(own)) {
                    vu = or8(vu, own);
                    st8(a.V, u, vu);
                }
                M8 want = andnot8(full, vu);  // sources that have not reached u
                const int beg = a.in_off[u], end = a.in_off[u + 1];
                if (any8(want) && beg < end) {
                    M8 acc = none8();
                    const int lim = min(end, beg + BU_INLINE);
                    int e = beg;
                    // four masks in flight (past the end: the list's first again)
                    for (; e < lim; e += 4) {
                        M8 f[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) f[k] = ld8(cur, a.in_adj[e + k < lim ? e + k : beg]);
                        acc = or8(acc, or8(or8(f[0], f[1]), or8(f[2], f[3])));
                        if (!any8(andnot8(want, acc))) break;
                    }
                    hard = e >= lim && lim < end;
                    pieces = hard && end - lim > LEVELS_PIECE ? (end - lim + LEVELS_PIECE - 1) / LEVELS_PIECE : 0;
                    const M8 nw = M8{make_uint4(acc.a.x & want.a.x, acc.a.y & want.a.y, acc.a.z & want.a.z, acc.a.w & want.a.w),
                                     make_uint4(acc.b.x & want.b.x, acc.b.y & want.b.y, acc.b.z & want.b.z, acc.b.w & want.b.w)};
                    if (any8(nw)) {
                        st8(next, u, nw);
                        found = true;
                        ++nf;
                        mf += a.off[u + 1] - a.off[u];
                    }
                }
            }
            const uint64_t fm = wave_ballot(found);
            const uint32_t mine = (lane < 32) ? (uint32_t)fm : (uint32_t)(fm >> 32);
            if ((lane & 31) == 0 && u < a.n) {  // each wave owns its 64 vertices' words
                if (mine) act_next[u >> 5] = mine;
                act_cur[u >> 5] = 0;  // (the next level's empty target)
            }
            int htot;
            const int hex = block_exclusive_scan<BLK>(hard && !pieces ? 1 : 0, s_w, &htot);
            if (htot > 0) {
                if (threadIdx.x == 0) s_hb = atomicAdd(&c->nhard, htot);
                __syncthreads();
                if (hard && !pieces) a.hard[s_hb + hex] = u;
                __syncthreads();
            }
            if (__syncthreads_or(pieces)) {
                int ptot;
                const int pex = block_exclusive_scan<BLK>(pieces, s_w, &ptot);
                if (threadIdx.x == 0) s_hb = atomicAdd(&c->nchunks, ptot);
                __syncthreads();
                const int beg = pieces ? a.in_off[u] + BU_INLINE : 0, end = pieces ? a.in_off[u + 1] : 0;
                for (int t = 0; t < pieces; ++t) {
                    const int64_t slot = (int64_t)s_hb + pex + t;
                    const int b = beg + t * LEVELS_PIECE;
                    if (slot < a.task_cap) a.tasks[slot] = ChunkRec{u, b, end - b > LEVELS_PIECE ? b + LEVELS_PIECE : end, 0};
                    else atomicOr(&c->changed, 1 << 30);
                }
                __syncthreads();
            }
        }
    }
    write_part<BLK>(a.fa, nf, mf, 0);
}

// OR of the masks of in-edges [beg, end) (whole wave, beg < end), until they cover `want`.
__device__ __forceinline__ M8 bl_gather(const LevelsArgs &a, const uint4 *cur, int beg, int end, const M8 &want) {
    const int lane = lane_id();
    M8 acc = none8();
    for (int e0 = beg; e0 < end; e0 += 4 * WAVE) {
        M8 f[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int e = e0 + k * WAVE + lane;
            f[k] = ld8(cur, a.in_adj[e < end ? e : beg]);
        }
        acc = or8(acc, or8(or8(f[0], f[1]), or8(f[2], f[3])));
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) acc = or8(acc, shfl_xor8(acc, o));
        if (!any8(andnot8(want, acc))) break;
    }
    return acc;
}

__global__ __launch_bounds__(BLK) void bl_b(LevelsArgs a) {
    Ctl *c = a.ctl;
    if (c->done) return;
    const int L = c->level;
    const uint4 *cur = a.level(L);
    uint4 *next = a.level(L + 1);
    uint32_t *act_next = a.act[(L + 1) & 1];
    const int lane = lane_id();
    const int wave = (blockIdx.x * BLK + (int)threadIdx.x) / WAVE, nwaves = gridDim.x * BLK / WAVE;
    long long nf = 0, mf = 0;
    if (c->dir == DIR_TD) {
        const int nt = (int)min((int64_t)c->nchunks, a.task_cap);
        for (int t = wave; t < nt; t += nwaves) {
            const ChunkRec r = a.tasks[t];
            const M8 fv = ld8(cur, r.v);
            for (int e = r.beg + lane; e < r.end; e += WAVE) bl_push(a, fv, a.adj[e], cur, next, act_next, nf, mf);
        }
    } else {
        const int nh = c->nhard;
        const M8 full = ld8(reinterpret_cast<const uint4 *>(a.sc->assigned), 0);
        for (int h = wave; h < nh; h += nwaves) {
            const int u = a.hard[h];
            const M8 prev = ld8(next, u);                          // bits found by the lane scan
            const M8 want = andnot8(andnot8(full, ld8(a.V, u)), prev);
            const M8 acc = bl_gather(a, cur, a.in_off[u] + BU_INLINE, a.in_off[u + 1], want);
            if (lane == 0) {
                const M8 nw = andnot8(want, andnot8(want, acc));
                if (any8(nw)) {
                    st8(next, u, or8(nw, prev));
                    if (!any8(prev)) {
                        atomicOr(&act_next[u >> 5], 1u << (u & 31));
                        ++nf;
                        mf += a.off[u + 1] - a.off[u];
                    }
                }
            }
        }
        const int np = (int)min((int64_t)c->nchunks, a.task_cap);
        for (int t = wave; t < np; t += nwaves) {
            const ChunkRec r = a.tasks[t];
            const int u = r.v;
            const M8 want = andnot8(andnot8(full, ld8(a.V, u)), ld8(next, u));  // (what other pieces added so far)
            if (!any8(want)) continue;
            const M8 acc = bl_gather(a, cur, r.beg, r.end, want);
            const M8 nw = andnot8(want, andnot8(want, acc));
            if (lane == 0 && any8(nw)) {
                uint32_t *nu = reinterpret_cast<uint32_t *>(next + 2 * (int64_t)u);
#pragma unroll
                for (int w = 0; w < 8; ++w)
                    if (word8(nw, w)) atomicOr(&nu[w], word8(nw, w));
                if (set_bit_first(act_next, u)) {
                    ++nf;
                    mf += a.off[u + 1] - a.off[u];
                }
            }
        }
    }
    write_part<BLK>(a.fa, nf, mf, 0);
    if (blockIdx.x == 0 && threadIdx.x == 0) c->pending = 1;
}

// The depths of vertex v (a lane each) from every level's mask, as P bit planes of the
// level number and the reached mask, then row by row: out[s * n + v].
template <int P>
__device__ __forceinline__ void bl_rows(const LevelsArgs &a, int levels, int u, int v, bool in, int k, int *out,
                                        long long &te, long long &nr) {
    uint32_t reached[8], plane[P][8];
#pragma unroll
    for (int w = 0; w < 8; ++w) {
        reached[w] = 0;
#pragma unroll
        for (int p = 0; p < P; ++p) plane[p][w] = 0;
    }
    for (int l = 0; l <= levels; ++l) {
        const M8 h = ld8(a.level(l), u);
#pragma unroll
        for (int w = 0; w < 8; ++w) {
            const uint32_t x = word8(h, w);
            reached[w] |= x;
#pragma unroll
            for (int p = 0; p < P; ++p) plane[p][w] |= (l >> p) & 1 ? x : 0u;
        }
    }
    if (!in) return;
    int cnt = 0;
#pragma unroll
    for (int w = 0; w < 8; ++w) cnt += __popc(reached[w]);
    nr += cnt;
    te += (long long)cnt * (a.off[u + 1] - a.off[u]);
#pragma unroll
    for (int w = 0; w < 8; ++w) {
        const int lim = min(32, k - 32 * w);
        int *row = out + (int64_t)32 * w * a.n + v;
        for (int b = 0; b < lim; ++b, row += a.n) {
            int d = 0;
#pragma unroll
            for (int p = 0; p < P; ++p) d |= (int)((plane[p][w] >> b) & 1u) << p;
            *row = (reached[w] >> b) & 1u ? d : -1;
        }
    }
}

// Every level as depths in the caller's order (perm: caller's id -> id here, or null).
__global__ __launch_bounds__(BLK) void bl_expand(LevelsArgs a, const int *perm, int k, int *out) {
    const int levels = a.ctl->level;
    long long te = 0, nr = 0;
    for (int base = blockIdx.x * BLK; base < a.n; base += gridDim.x * BLK) {
        const int v = base + (int)threadIdx.x;
        const bool in = v < a.n;
        const int u = in ? (perm ? perm[v] : v) : 0;
        if (levels < 8) bl_rows<3>(a, levels, u, v, in, k, out, te, nr);
        else if (levels < 16) bl_rows<4>(a, levels, u, v, in, k, out, te, nr);
        else bl_rows<5>(a, levels, u, v, in, k, out, te, nr);
    }
    te = block_sum<BLK>(te);
    nr = block_sum<BLK>(nr);
    if (threadIdx.x == 0) {
        atomicAdd((unsigned long long *)&a.ctl->edges_traversed, (unsigned long long)te);
        atomicAdd((unsigned long long *)&a.ctl->reached, (unsigned long long)nr);
    }
}

// Runs a batched BFS on the graph's context b by levels; *deep is set (and nothing
// delivered) when the search is too deep for them.  perm as in bl_expand.
int bfs_levels_run(mg_graph *g, BatchDev &b, const int32_t *slot_of, const int32_t *srcs, int32_t npairs, int32_t k,
                   int32_t *depth_out, const mg_options &o, mg_stats *stats, const CallTimer &timer, bool *deep) {
    int rc;
    *deep = false;
    LevelsArgs a{};
    a.ctl = b.ctl;
    a.sc = b.sc;
    a.off = g->row_off;
    a.adj = g->col;
    if (g->flags & MG_GRAPH_SYMMETRIC) {
        a.in_off = g->row_off;
        a.in_adj = g->col;
    } else if (g->col_off) {
        a.in_off = g->col_off;
        a.in_adj = g->row_idx;
    }
    a.V = b.V;
    a.H = reinterpret_cast<uint4 *>(b.rows);
    a.act[0] = b.act[0];
    a.act[1] = b.act[1];
    a.hard = b.hard;
    a.tasks = b.tasks;
    a.task_cap = b.task_cap;
    a.fa.part = b.part;
    a.n = g->n;
    a.nwords = b.nwords;
    a.G = b.G;
    // the result: the caller's device buffer, else rows of our own
    int *out = depth_out;
    if (!plan_delivery(g, depth_out, 4 * (size_t)k * g->n, o.out_on_device).by_kernel) {
        const int64_t cells = (int64_t)k * g->n;
        if (!g->perm && b.rows_out_cap < cells) {  // (a twin's context has rows for every slot)
            free_dev(b.rows_out);
            b.rows_out = nullptr;
            b.bytes -= 4 * b.rows_out_cap;
            b.rows_out_cap = 0;
            if ((rc = alloc_i32(&b.rows_out, (size_t)cells))) return rc;
            b.rows_out_cap = cells;
            b.bytes += 4 * cells;
        }
        out = b.rows_out;
    }
    MG_HIP(hipEventRecord(g->ev0, g->stream));
    hipLaunchKernelGGL(bl_init, dim3(grid_blocks(4 * (int64_t)g->n, BLK)), dim3(BLK), 0, g->stream, a, o.iter_num,
                       a.in_off != nullptr, o.batch_alpha > 0 ? o.batch_alpha : LEVELS_ALPHA, batch_beta(o),
                       (long long)g->m);
    for (int i0 = 0; i0 < npairs; i0 += MG_BATCH_MAX) {
        SeedList sl{};
        for (int i = i0; i < npairs && i < i0 + MG_BATCH_MAX; ++i) {
            sl.slot[sl.n] = slot_of[i];
            sl.src[sl.n++] = srcs[i];
        }
        hipLaunchKernelGGL(bl_seed, dim3(1), dim3(MG_BATCH_MAX), 0, g->stream, a, sl);
    }
    MG_HIP(hipGetLastError());
    auto step = [&]() -> int {
        hipLaunchKernelGGL(bl_close, dim3(1), dim3(SMALL_BLK), 0, g->stream, a);
        hipLaunchKernelGGL(bl_a, dim3(a.G), dim3(BLK), 0, g->stream, a);
        hipLaunchKernelGGL(bl_b, dim3(a.G), dim3(BLK), 0, g->stream, a);
        MG_HIP(hipGetLastError());
        return MG_OK;
    };
    if ((rc = drive(g, step, LEVELS_MAX + 2, KIND_BATCH, 1, b.ctl, b.h_ctl))) return rc;
    if (b.h_ctl->changed & (1 << 30))
        return set_error(MG_ERR_OVERFLOW, "batched task queue overflow (capacity %lld)", (long long)b.task_cap);
    if (b.h_ctl->changed & LEVELS_DEEP) {
        *deep = true;
        return MG_OK;
    }
    hipLaunchKernelGGL(bl_expand, dim3(grid_blocks_cap(g->n, BLK, 4 * MAX_GRID)), dim3(BLK), 0, g->stream, a,
                       (const int *)g->perm, k, out);
    MG_HIP(hipGetLastError());
    MG_HIP(hipEventRecord(g->ev1, g->stream));
    MG_HIP(hipMemcpyAsync(b.h_ctl, b.ctl, sizeof(Ctl), hipMemcpyDeviceToHost, g->stream));
    MG_HIP(hipStreamSynchronize(g->stream));
    float ms = 0;
    MG_HIP(hipEventElapsedTime(&ms, g->ev0, g->ev1));
    if (stats) {
        std::memset(stats, 0, sizeof *stats);
        stats->iterations = b.h_ctl->level;
        stats->bottom_up_levels = b.h_ctl->bu_levels;
        stats->edges_examined = b.h_ctl->edges_examined;
        stats->edges_traversed = b.h_ctl->edges_traversed;
        stats->vertices_reached = b.h_ctl->reached;
        stats->device_ms = ms;
    }
    if (out != depth_out && (rc = deliver(g, depth_out, out, 4 * (size_t)k * g->n, o.out_on_device))) return rc;
    if (stats) stats->host_ms = timer.ms();
    return MG_OK;
}

}  // namespace mg
