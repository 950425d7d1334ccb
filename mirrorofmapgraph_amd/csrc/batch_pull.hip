// Batched SSSP by pulling: the path of mg_sssp_batch on graphs of mean degree 8 and more
// with an in-edge view.
//
// batch_sssp.hip pushes: for every edge of a frontier vertex a wave relaxes all slots with
// an atomicMin per improvement and ORs the pair masks.  On power-law graphs a few dense
// rounds are nearly all of the work, and every vertex is a target of many relaxations.  Here
// a group of lanes (four slots each) owns a vertex for the round, keeps its row of distances
// in registers, takes the minimum over its in-edges of the neighbour's row + weight and
// stores the row once: no atomics, no masks, no buckets (long in-lists, cut into pieces, are
// merged with atomicMin).  One launch and a close per round.
//
// What keeps the rounds short are two numbers per vertex: `low`, the smallest distance that
// changed there in the last round (INT_MAX: none did), and `top`, a bound on the largest
// distance of its row.  An edge (v, u, w) can only improve u when low[v] + w < top[u], so
// the rows (16 bytes a lane) are touched only then: a wave first streams the edges of its
// task, a lane each, with one 4-byte gather from an array that stays in the L2, and keeps
// the edges that pass in LDS, in order; then its groups take the vertices that have any.
// Only slots that changed somewhere in the last round count for `top`: the others are
// settled (a source in a small component leaves most vertices unreached, and would make
// the test useless).
//
// A row read while its owner stores it is a mix of old and new distances, each an upper
// bound; the change puts `low` up for the next round.  Rounds end when nothing changed, so
// every slot has its unique shortest distances.  A search of more than PULL_ROUNDS rounds
// (a mesh with many neighbours) stops and is run again the pushing way, as are all later
// ones on the graph.
//
// Bound by the row gathers of the dense rounds: 250,001 vertices, m = 7.65 M, 100 sources:
// about 4.3 m rows of 400 bytes in all, 6 TB/s (the 128 MB of rows fit the Infinity Cache).
// 9.35 ms pushing (7.8 after its slices fitted the graph), 2.65 here; 4.1 ms with a group per vertex
// reading its list and its row before the test (rounds that change nothing took 125 us, now
// 40).
#include <climits>
#include <vector>

#include "batch.h"

namespace mg {

constexpr int PULL_ROUNDS = 48;
constexpr int PULL_DEEP = 1 << 29;        // Ctl::changed: too many rounds
constexpr int64_t PULL_DEGREE = 8;
constexpr int PULL_T = 512;               // in-edges of a wave task

struct PullArgs {
    Ctl *ctl;
    FrontierArgs fa;          // level counters only (part)
    const int *in_off, *in_adj, *eid, *w, *off;
    const ChunkRec *tasks;    // wave tasks: {v0, -, -, vertices} or a piece {v, beg, end, 0}
    int ntasks, n, k;
    int wmin;                 // smallest edge weight
    int *D;                   // n rows of 4 * LANES distances; slots past k hold 0
    int *low[3];              // by round % 3
    int *top;
    uint32_t *live;           // 3 x 8 words, by round % 3: slots that changed
};

// Device state of a graph's pulled batches.
struct PullDev {
    Ctl *ctl = nullptr, *h_ctl = nullptr;
    LevelPart *part = nullptr;
    uint32_t *live = nullptr;
    int *low = nullptr;       // low (3 n) and top (n)
    ChunkRec *tasks = nullptr;
    int ntasks = 0;
    int *D = nullptr, *rows = nullptr;
    int64_t d_cap = 0, rows_cap = 0;
};

// Rows of INT_MAX (0 past slot k), nothing changed, every slot live.
__global__ void pull_init(PullArgs a, int lanes, int iter_limit) {
    const int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, nt = (int64_t)gridDim.x * blockDim.x;
    int4 *D4 = reinterpret_cast<int4 *>(a.D);
    for (int64_t i = tid; i < (int64_t)a.n * lanes; i += nt) {
        const int s = 4 * (int)(i % lanes);
        D4[i] = make_int4(s < a.k ? INT_MAX : 0, s + 1 < a.k ? INT_MAX : 0, s + 2 < a.k ? INT_MAX : 0,
                          s + 3 < a.k ? INT_MAX : 0);
    }
    for (int64_t i = tid; i < 4LL * a.n; i += nt) a.low[0][i] = INT_MAX;  // low and top
    if (blockIdx.x != 0) return;
    clear_parts(a.fa);
    if (threadIdx.x < 24) a.live[threadIdx.x] = threadIdx.x < 8 ? ~0u : 0u;
    if (threadIdx.x != 0) return;
    ctl_reset(a.ctl, a.n, iter_limit, 1);
    a.ctl->fmin = 0;
    a.ctl->aux = a.k;
}

__global__ void pull_seed(PullArgs a, int lanes, SeedList sl) {
    const int i = threadIdx.x;
    if (i >= sl.n) return;
    a.D[(int64_t)sl.src[i] * 4 * lanes + sl.slot[i]] = 0;
    a.low[0][sl.src[i]] = 0;
}

__global__ __launch_bounds__(SMALL_BLK) void pull_close(PullArgs a) {
    Ctl *c = a.ctl;
    if (c->done) return;
    if (threadIdx.x == 0) c->steps++;
    if (!c->pending) return;
    long long nf, mf, ex, mn;
    take_level_parts<SMALL_BLK>(a.fa, nf, mf, ex, &mn);
    const int L = c->level;
    if (threadIdx.x < 8) a.live[8 * ((L + 2) % 3) + threadIdx.x] = 0;  // round L + 1 sets these
    __syncthreads();
    if (threadIdx.x != 0) return;
    c->edges_examined += ex;
    c->fmin = mn;
    c->pending = 0;
    c->level = L + 1;
    c->nf_prev = (int)nf;
    if (nf == 0 || L + 1 >= c->iter_limit) {
        c->done = 1;
    } else if (L + 1 >= PULL_ROUNDS) {
        c->changed |= PULL_DEEP;
        c->done = 1;
    }
}

// x reduced over the group of LANES lanes that this lane belongs to (every lane gets it).
template <int LANES, class Op>
__device__ __forceinline__ int group_reduce(int x, Op op) {
#pragma unroll
    for (int o = LANES / 2; o > 0; o >>= 1) x = op(x, __shfl_xor(x, o));
    return x;
}

// The largest distance of a row over the live slots, in every lane of its group.
template <int LANES>
__device__ __forceinline__ int row_top(const uint4 &cur, const uint4 &on) {
    const uint32_t x = max(max(cur.x & on.x, cur.y & on.y), max(cur.z & on.z, cur.w & on.w));
    return group_reduce<LANES>((int)x, [](int p, int q) { return max(p, q); });
}

// A wave's edges that pass the test, in order, and the vertices of its task.
struct PullLds {
    int v[PULL_T], w[PULL_T];
    unsigned char own[PULL_T];  // vertex of the task
    short seg[WAVE + 1];        // first edge of each vertex that has any
    int off[WAVE + 1], top[WAVE], low[WAVE];
};

// cur becomes the minimum of itself and the rows of the kept edges [p, end) plus weight;
// four rows a step (every lane of the wave calls it, each group with its own range).
template <int LANES>
__device__ __forceinline__ void pull_rows_min(const PullArgs &a, const PullLds &q, int p, int end, bool used,
                                              uint4 &cur) {
    const uint4 *D4 = reinterpret_cast<const uint4 *>(a.D);
    const int gl = lane_id() % LANES;
    for (; wave_ballot(p < end); p += 4) {
        uint4 row[4];
        uint32_t ws[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = p + j < end ? p + j : 0;  // (past the end: edge 0's row, ignored)
            ws[j] = p + j < end ? (uint32_t)q.w[i] : ~0u;
            row[j] = make_uint4(0, 0, 0, 0);
            if (used) row[j] = D4[(int64_t)q.v[i] * LANES + gl];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (ws[j] == ~0u) continue;
            // unsigned: an unreached INT_MAX plus a weight does not wrap
            cur.x = min(cur.x, row[j].x + ws[j]);
            cur.y = min(cur.y, row[j].y + ws[j]);
            cur.z = min(cur.z, row[j].z + ws[j]);
            cur.w = min(cur.w, row[j].w + ws[j]);
        }
    }
}

// One round: a wave per task.
template <int LANES, bool EID>
__global__ __launch_bounds__(BLK) void pull_round(PullArgs a) {
    Ctl *c = a.ctl;
    if (c->done) return;
    constexpr int GROUPS = WAVE / LANES;
    __shared__ PullLds s_q[BLK / WAVE];
    __shared__ uint32_t s_moved[8];
    const int L = c->level, lane = lane_id(), gl = lane % LANES, grp = lane / LANES, wv = (int)threadIdx.x / WAVE;
    PullLds &q = s_q[wv];
    const int *low = a.low[L % 3];
    int *low_next = a.low[(L + 1) % 3], *low_clear = a.low[(L + 2) % 3];
    uint4 *D4 = reinterpret_cast<uint4 *>(a.D);
    const bool used = 4 * gl < c->aux;  // (a.k is the capturing call's)
    // this lane's live slots, as masks over their distances
    const uint32_t lw = a.live[8 * (L % 3) + gl / 8] >> (4 * (gl % 8));
    const uint4 on = make_uint4(lw & 1 ? ~0u : 0u, lw & 2 ? ~0u : 0u, lw & 4 ? ~0u : 0u, lw & 8 ? ~0u : 0u);
    // a distance changed in the last round is at least fmin: rows up to this stay as they are
    const int least = (int)min(c->fmin + a.wmin, (long long)INT_MAX);
    long long nf = 0, ex = 0, mn = LLONG_MAX;
    uint32_t moved = 0;  // this lane's slots that changed somewhere
    if (threadIdx.x < 8) s_moved[threadIdx.x] = 0;
    const int wave = (blockIdx.x * BLK + (int)threadIdx.x) / WAVE, nwaves = gridDim.x * BLK / WAVE;
    for (int t = wave; t < a.ntasks; t += nwaves) {
        const ChunkRec r = a.tasks[t];
        const bool piece = r.pad == 0;
        const int va = r.v, nv = piece ? 1 : r.pad;
        const int beg = piece ? r.beg : a.in_off[va + min(lane, nv)];
        const int topv = lane < nv ? a.top[va + lane] : 0;
        if (!wave_ballot(topv > least)) {  // no edge can improve any of the rows
            if (lane < nv) (piece ? low_clear : low_next)[va + lane] = INT_MAX;
            continue;
        }
        q.off[lane] = beg;
        q.top[lane] = topv;
        q.low[lane] = INT_MAX;
        const int e0 = __builtin_amdgcn_readfirstlane(beg);
        const int e1 = piece ? r.end : a.in_off[va + nv];
        wave_sync();
        // the edges that pass, 4 x 64 at a time
        int cnt = 0;
        for (int eb = e0; eb < e1; eb += 4 * WAVE) {
            int v[4], wt[4], own[4], lo[4];
            bool ok[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int e = eb + j * WAVE + lane;
                ok[j] = e < e1;
                const int sl = ok[j] ? e : e0;
                v[j] = a.in_adj[sl];
                wt[j] = EID ? a.eid[sl] : a.w[sl];
                own[j] = 0;  // the last vertex whose list starts at or before the edge
                if (!piece) {
#pragma unroll
                    for (int st = WAVE / 2; st > 0; st >>= 1)
                        if (own[j] + st < nv && q.off[own[j] + st] <= sl) own[j] += st;
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (EID) wt[j] = a.w[wt[j]];
                lo[j] = low[v[j]];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool need = ok[j] && lo[j] < q.top[own[j]] - wt[j];
                const uint64_t m = wave_ballot(need);
                if (need) {
                    const int i = cnt + lanes_below(m);
                    q.v[i] = v[j];
                    q.w[i] = wt[j];
                    q.own[i] = (unsigned char)own[j];
                }
                cnt += __popcll(m);
            }
        }
        wave_sync();
        if (lane == 0) ex += cnt;
        if (piece) {
            if (lane == 0) low_clear[va] = INT_MAX;
            if (cnt == 0) continue;
            // the groups share the kept edges and merge their minima
            const uint4 old = used ? D4[(int64_t)va * LANES + gl] : make_uint4(0, 0, 0, 0);
            uint4 cur = old;
            const int per = (cnt + GROUPS - 1) / GROUPS;
            pull_rows_min<LANES>(a, q, grp * per, min(grp * per + per, cnt), used, cur);
#pragma unroll
            for (int o = LANES; o < WAVE; o <<= 1) {
                cur.x = min(cur.x, (uint32_t)__shfl_xor((int)cur.x, o));
                cur.y = min(cur.y, (uint32_t)__shfl_xor((int)cur.y, o));
                cur.z = min(cur.z, (uint32_t)__shfl_xor((int)cur.z, o));
                cur.w = min(cur.w, (uint32_t)__shfl_xor((int)cur.w, o));
            }
            const uint32_t ch = (cur.x < old.x) | (cur.y < old.y) << 1 | (cur.z < old.z) << 2 | (cur.w < old.w) << 3;
            int lo = INT_MAX;
            if (ch & 1) lo = min(lo, (int)cur.x);
            if (ch & 2) lo = min(lo, (int)cur.y);
            if (ch & 4) lo = min(lo, (int)cur.z);
            if (ch & 8) lo = min(lo, (int)cur.w);
            lo = group_reduce<WAVE>(lo, [](int x, int y) { return min(x, y); });
            const int top = row_top<LANES>(cur, on);
            moved |= ch;
            if (grp == 0) {
                int *d = a.D + 4 * ((int64_t)va * LANES + gl);
                if (ch & 1) atomicMin(d, (int)cur.x);
                if (ch & 2) atomicMin(d + 1, (int)cur.y);
                if (ch & 4) atomicMin(d + 2, (int)cur.z);
                if (ch & 8) atomicMin(d + 3, (int)cur.w);
            }
            if (lane == 0) {
                if (top < topv) atomicMin(&a.top[va], top);  // (other pieces only lower the row)
                if (lo != INT_MAX) {
                    atomicMin(&low_next[va], lo);
                    ++nf;
                    mn = min(mn, (long long)lo);
                }
            }
            continue;
        }
        // the vertices with edges left: a group each
        int ns = 0;
        for (int p0 = 0; p0 < cnt; p0 += WAVE) {
            const int p = p0 + lane;
            const bool head = p < cnt && (p == 0 || q.own[p] != q.own[p - 1]);
            const uint64_t m = wave_ballot(head);
            if (head) q.seg[ns + lanes_below(m)] = (short)p;
            ns += __popcll(m);
        }
        if (lane == 0) q.seg[ns] = (short)cnt;
        wave_sync();
        for (int s0 = 0; s0 < ns; s0 += GROUPS) {
            const bool mine = s0 + grp < ns;
            const int p = mine ? q.seg[s0 + grp] : 0, end = mine ? q.seg[s0 + grp + 1] : 0;
            const int own = q.own[p];
            const int64_t at = (int64_t)(va + own) * LANES + gl;
            const uint4 old = used ? D4[at] : make_uint4(0, 0, 0, 0);
            uint4 cur = old;
            pull_rows_min<LANES>(a, q, p, end, used, cur);
            const uint32_t ch = (cur.x < old.x) | (cur.y < old.y) << 1 | (cur.z < old.z) << 2 | (cur.w < old.w) << 3;
            int lo = INT_MAX;
            if (ch & 1) lo = min(lo, (int)cur.x);
            if (ch & 2) lo = min(lo, (int)cur.y);
            if (ch & 4) lo = min(lo, (int)cur.z);
            if (ch & 8) lo = min(lo, (int)cur.w);
            lo = group_reduce<LANES>(lo, [](int x, int y) { return min(x, y); });
            const int top = row_top<LANES>(cur, on);
            if (mine && ch) {
                D4[at] = cur;
                moved |= ch;
            }
            if (mine && gl == 0) {
                a.top[va + own] = top;
                if (lo != INT_MAX) {
                    q.low[own] = lo;
                    ++nf;
                    mn = min(mn, (long long)lo);
                }
            }
        }
        wave_sync();
        if (lane < nv) low_next[va + lane] = q.low[lane];
        wave_sync();  // the next task rewrites this wave's LDS
    }
    __syncthreads();
    if (moved) atomicOr(&s_moved[gl / 8], moved << (4 * (gl % 8)));
    __syncthreads();
    if (threadIdx.x < 8) {
        uint32_t *p = &a.live[8 * ((L + 1) % 3) + threadIdx.x];
        const uint32_t add = s_moved[threadIdx.x];
        if (add & ~(uint32_t)ld_dev((const int *)p)) atomicOr(p, add);
    }
    write_part<BLK>(a.fa, nf, 0, ex, mn);
    if (blockIdx.x == 0 && threadIdx.x == 0) c->pending = 1;
}

// Distances as rows in the caller's order (perm: caller's id -> id here, or null), 64
// vertices x 64 slots through LDS, with the TEPS count and the reached vertices.
__global__ __launch_bounds__(BLK) void pull_rows(PullArgs a, int ks, const int *perm, int *out) {
    __shared__ int tile[64][65];
    long long te = 0, nr = 0;
    const int tv = (a.n + 63) / 64, ts = (a.k + 63) / 64;
    for (int t = blockIdx.x; t < tv * ts; t += gridDim.x) {
        const int v0 = (t % tv) * 64, s0 = (t / tv) * 64;
        for (int i = threadIdx.x; i < 64 * 64; i += BLK) {
            const int r = i / 64, cc = i % 64, v = v0 + r, s = s0 + cc;
            // a wave reads 64 slots of one vertex
            const int u = v < a.n ? (perm ? perm[v] : v) : 0;
            const int d = v < a.n && s < a.k ? a.D[(int64_t)u * ks + s] : INT_MAX;
            tile[r][cc] = d;
            const int reached = __popcll(wave_ballot(d != INT_MAX));
            if (cc == 0 && reached) {
                nr += reached;
                te += (long long)reached * (a.off[u + 1] - a.off[u]);
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < 64 * 64; i += BLK) {
            const int cc = i / 64, r = i % 64, v = v0 + r, s = s0 + cc;
            if (v < a.n && s < a.k) out[(int64_t)s * a.n + v] = tile[r][cc];
        }
        __syncthreads();
    }
    te = block_sum<BLK>(te);
    nr = block_sum<BLK>(nr);
    if (threadIdx.x == 0) {
        if (te) atomicAdd((unsigned long long *)&a.ctl->edges_traversed, (unsigned long long)te);
        if (nr) atomicAdd((unsigned long long *)&a.ctl->reached, (unsigned long long)nr);
    }
}

// ---------------------------------------------------------------- host side

// The captured rounds, which point at the state's buffers.
static void pull_drop_steps(mg_graph *g) {
    for (int w = 0; w < 4; ++w) invalidate_steps(g, KIND_BATCH_PULL + w);
}

void pull_release(mg_graph *g) {
    PullDev *&p = g->steps->pull;
    if (!p) return;
    pull_drop_steps(g);
    free_dev(p->ctl);
    if (p->h_ctl) (void)hipHostFree(p->h_ctl);
    free_dev(p->part);
    free_dev(p->live);
    free_dev(p->low);
    free_dev(p->tasks);
    free_dev(p->D);
    free_dev(p->rows);
    delete p;
    p = nullptr;
    g->steps->pull_bytes = 0;
}

bool pull_wanted(const mg_graph *g) {
    return g->m >= PULL_DEGREE * (int64_t)g->n && ((g->flags & MG_GRAPH_SYMMETRIC) || g->col_off) &&
           !g->steps->pull_deep;
}

// The wave tasks over the in-lists: runs of consecutive vertices with at most PULL_T
// in-edges in all (and at most a vertex per lane), and pieces of the longer lists.
static int pull_tasks(mg_graph *g, PullDev &p, const int *d_in_off) {
    const int n = g->n;
    std::vector<int32_t> off((size_t)n + 1);
    MG_HIP(copy_on(g->stream, off.data(), d_in_off, 4 * ((size_t)n + 1), hipMemcpyDeviceToHost));
    std::vector<ChunkRec> t;
    for (int v = 0; v < n;) {
        if (off[v + 1] - off[v] > PULL_T) {
            for (int b = off[v]; b < off[v + 1]; b += PULL_T) t.push_back(ChunkRec{v, b, std::min(b + PULL_T, off[v + 1]), 0});
            ++v;
            continue;
        }
        int u = v + 1;
        while (u < n && u - v < WAVE && off[u + 1] - off[v] <= PULL_T) ++u;
        t.push_back(ChunkRec{v, 0, 0, u - v});
        v = u;
    }
    int rc = alloc_chunks(&p.tasks, t.size());
    if (rc) return rc;
    if (!t.empty() &&
        copy_on(g->stream, p.tasks, t.data(), sizeof(ChunkRec) * t.size(), hipMemcpyHostToDevice) != hipSuccess)
        return set_error(MG_ERR_DEVICE, "task copy failed");
    p.ntasks = (int)t.size();
    g->steps->pull_bytes += (int64_t)(sizeof(ChunkRec) * t.size());
    return MG_OK;
}

template <int LANES>
static void launch_round(const PullArgs &a, int blocks, hipStream_t st) {
    if (a.eid) hipLaunchKernelGGL((pull_round<LANES, true>), dim3(blocks), dim3(BLK), 0, st, a);
    else hipLaunchKernelGGL((pull_round<LANES, false>), dim3(blocks), dim3(BLK), 0, st, a);
}

int pull_batch(mg_graph *g, const int32_t *row_of, const int32_t *srcs, int32_t npairs, int32_t k, int32_t *out,
               const mg_options &o, mg_stats *stats, const CallTimer &timer, bool *deep) {
    int rc;
    *deep = false;
    const bool sym = g->flags & MG_GRAPH_SYMMETRIC;
    const int *in_off = sym ? g->row_off : g->col_off;
    PullDev *&pp = g->steps->pull;
    if (!pp && !(pp = new (std::nothrow) PullDev())) return set_error(MG_ERR_OOM, "host allocation failed");
    PullDev &p = *pp;
    const int lanes = pull_lanes(k), ks = 4 * lanes;
    if (!p.ctl) {
        int *c = nullptr, *l = nullptr;
        if ((rc = alloc_i32(&c, sizeof(Ctl) / 4)) || (rc = alloc_parts(&p.part, PART_GROUPS)) ||
            (rc = alloc_i32(&l, 24)) || (rc = alloc_i32(&p.low, 4 * (size_t)g->n)) || (rc = pull_tasks(g, p, in_off)) ||
            hipHostMalloc((void **)&p.h_ctl, sizeof(Ctl), hipHostMallocDefault) != hipSuccess) {
            free_dev(c);
            free_dev(l);
            pull_release(g);
            return rc ? rc : set_error(MG_ERR_OOM, "hipHostMalloc failed");
        }
        p.ctl = reinterpret_cast<Ctl *>(c);
        p.live = reinterpret_cast<uint32_t *>(l);
        g->steps->pull_bytes += (int64_t)sizeof(Ctl) + (int64_t)sizeof(LevelPart) * PART_GROUPS + 96 + 16LL * g->n;
    }
    const bool direct = plan_delivery(g, out, 4 * (size_t)k * g->n, o.out_on_device).by_kernel;
    auto grow = [&](int **buf, int64_t *cap, int64_t need) -> int {
        if (*cap >= need) return MG_OK;
        MG_HIP(hipStreamSynchronize(g->stream));
        pull_drop_steps(g);
        free_dev(*buf);
        *buf = nullptr;
        g->steps->pull_bytes -= 4 * *cap;
        *cap = 0;
        const int arc = alloc_i32(buf, (size_t)need);
        if (arc) return arc;
        *cap = need;
        g->steps->pull_bytes += 4 * need;
        return MG_OK;
    };
    if ((rc = grow(&p.D, &p.d_cap, (int64_t)ks * g->n))) return rc;
    if (!direct && (rc = grow(&p.rows, &p.rows_cap, (int64_t)k * g->n))) return rc;
    PullArgs a{};
    a.ctl = p.ctl;
    a.fa.part = p.part;
    a.in_off = in_off;
    a.in_adj = sym ? g->col : g->row_idx;
    a.eid = sym ? nullptr : g->csc_eid;
    a.w = g->w;
    a.wmin = g->min_weight;
    a.off = g->row_off;
    a.tasks = p.tasks;
    a.ntasks = p.ntasks;
    a.top = p.low + 3 * (size_t)g->n;
    a.n = g->n;
    a.k = k;
    a.D = p.D;
    for (int i = 0; i < 3; ++i) a.low[i] = p.low + (size_t)i * g->n;
    a.live = p.live;
    MG_HIP(hipEventRecord(g->ev0, g->stream));
    hipLaunchKernelGGL(pull_init, dim3(grid_blocks_cap((int64_t)g->n * lanes, BLK, 4 * MAX_GRID)), dim3(BLK), 0,
                       g->stream, a, lanes, o.iter_num);
    for (int i0 = 0; i0 < npairs; i0 += MG_BATCH_MAX) {
        SeedList sl{};
        for (int i = i0; i < npairs && i < i0 + MG_BATCH_MAX; ++i) {
            sl.slot[sl.n] = row_of[i];
            sl.src[sl.n++] = srcs[i];
        }
        hipLaunchKernelGGL(pull_seed, dim3(1), dim3(MG_BATCH_MAX), 0, g->stream, a, lanes, sl);
    }
    MG_HIP(hipGetLastError());
    const int blocks = grid_blocks_cap((int64_t)a.ntasks * WAVE, BLK, 8 * MAX_GRID);
    auto step = [&]() -> int {
        hipLaunchKernelGGL(pull_close, dim3(1), dim3(SMALL_BLK), 0, g->stream, a);
        switch (lanes) {
        case 8: launch_round<8>(a, blocks, g->stream); break;
        case 16: launch_round<16>(a, blocks, g->stream); break;
        case 32: launch_round<32>(a, blocks, g->stream); break;
        default: launch_round<64>(a, blocks, g->stream); break;
        }
        MG_HIP(hipGetLastError());
        return MG_OK;
    };
    const StepKey sk = batch_pull_steps(k);
    if ((rc = drive(g, step, PULL_ROUNDS + 2, sk.kind, sk.key, p.ctl, p.h_ctl))) return rc;
    if (p.h_ctl->changed & PULL_DEEP) {
        g->steps->pull_deep = *deep = true;
        pull_release(g);  // not taken again
        return MG_OK;
    }
    int *dst = direct ? out : p.rows;
    const int tiles = ((g->n + 63) / 64) * ((k + 63) / 64);
    hipLaunchKernelGGL(pull_rows, dim3(std::max(1, std::min(tiles, 4 * MAX_GRID))), dim3(BLK), 0, g->stream, a, ks,
                       (const int *)g->perm, dst);
    MG_HIP(hipGetLastError());
    MG_HIP(hipEventRecord(g->ev1, g->stream));
    MG_HIP(hipMemcpyAsync(p.h_ctl, p.ctl, sizeof(Ctl), hipMemcpyDeviceToHost, g->stream));
    MG_HIP(hipStreamSynchronize(g->stream));
    float ms = 0;
    MG_HIP(hipEventElapsedTime(&ms, g->ev0, g->ev1));
    if (stats) {
        std::memset(stats, 0, sizeof *stats);
        stats->iterations = p.h_ctl->level;
        stats->edges_examined = p.h_ctl->edges_examined;
        stats->edges_traversed = p.h_ctl->edges_traversed;
        stats->vertices_reached = p.h_ctl->reached;
        stats->device_ms = ms;
    }
    if (!direct && (rc = deliver(g, out, p.rows, 4 * (size_t)k * g->n, o.out_on_device))) return rc;
    if (stats) stats->host_ms = timer.ms();
    return MG_OK;
}

}  // namespace mg
