// Batched personalized PageRank: up to 64 sources (slots) iterate together.
//
// Not in the reference, whose PageRank (Algorithms/PageRank/PageRank.h:233-283) has
// one global teleport term; this is its personalized form, with the reference's
// conventions: contribution r[v] / outdeg(v) gathered over in-edges, rank-sink
// (dangling) mass dropped, teleport t applied as written there (t + (1 - t) * sum):
//   x_0 = e_s,   x_{i+1}[u] = (1 - t) * sum_{v -> u} x_i[v] / outdeg(v)  (+ t when u = s).
// Ranks are vertex-major, X[v * W + slot], W = 8, 16, 32 or 64 floats per vertex: the
// smallest width above every slot in use (slots are handed out lowest first; the rows
// are repacked when it changes), so a wave gathers the rows of 256 / W in-edges
// at a time and a row is one 32-byte sector while at most 8 slots are in use.
// Vertices are covered by static tasks: runs of consecutive vertices with at most
// ppr_piece() in-edges in total (one wave walks them), and pieces of that size of longer
// in-lists whose partial sums are added in piece order.  Every list is summed in one
// order fixed by the list alone, whatever the width (see team_list), so a slot's
// arithmetic is fixed by the graph: a query gives the same bits alone or beside any
// other queries.
#include "batch.h"

#include <vector>

namespace mg {

// In-edges per task: m / PPR_PIECES within these limits, so that small graphs have tasks for
// every wave (scale 16: 26 us an iteration with 1024 edges whatever the size, 17 so) and large
// ones as few pieces as fill the GPU (scale 20: 512 edges 208 us, 1024 174, 2048 172).
constexpr int PPR_PIECES = 16384, PPR_T_MIN = 256, PPR_T_MAX = 1024;
constexpr int PPR_RUN = 64;    // vertices per run task

struct PprArgs {
    const int *in_off, *in_adj;  // in-edges (CSR of a symmetric graph, or the CSC)
    const int *out_off;          // out-degrees
    const float *X;              // ranks, n x W (ppr_contrib)
    const float *C;              // contributions rank / outdeg, n x W, and a row of zeros
    float *D;                    // next contributions, or the ranks after the last iteration
    float *part;                 // piece partial sums, npart x W
    const ChunkRec *tasks;       // pieces of long lists: {v, beg, end, list}; then runs: {v0, -, -, count}
    int *big;                    // per long list: vertex, first part, parts, parts summed (4 ints)
    const int *src;              // per slot: source or -1
    int64_t m;
    int n, npart, ntasks;
    int last;                    // D takes ranks
    float t;                     // teleport
};

// Row width: ranks, contributions and partial sums are stored n x W, W the smallest
// of 8, 16, 32, 64 above every slot in use (slots are handed out lowest first), so a
// gathered row is W floats: 32 bytes (one sector) while at most 8 slots are in use,
// and the contribution array of a 4M-vertex graph is 128 MB instead of 1 GB.

// What bounds an iteration is reading rows that the L2 does not hold: at R-MAT scale 20 (31.4M
// edges) and W = 8, 29M lines of 128 bytes go from L2 to L1 (92 us at 64 bytes a clock and CU)
// and 6.4M from memory to the L2 (4.5 TB/s), at W = 64 4.7 GB (6.4 TB/s).  Below that the
// address unit is: it takes a quad of lanes a clock whatever the lanes load, so a lane loads
// four columns (16 bytes) at once, and four sources.  Four columns, a list per group and one
// launch an iteration, against a column per lane, a list per wave and three launches, us an
// iteration on the degree-ordered twin:
//   scale    W = 8         16          64
//   16     56 -> 17    76 -> 20    159 -> 53
//   18     99 -> 44   136 -> 57    312 -> 164
//   20    241 -> 174  378 -> 231  1070 -> 776
// Rows of the highest degrees kept in LDS took 185 at W = 8; the next block's sources loaded
// ahead of the gathers 185 (more registers, fewer waves).

// A wave's lanes for rows of W columns: V columns a lane, L lanes a row, G rows side by side.
// Eight partial sums make a list (see below): a team of T groups sums a list together, J
// partial sums a lane, NT teams a wave.
template <int W>
struct PprLanes {
    static constexpr int V = 4, L = W / V, G = WAVE / L, T = G < 8 ? G : 8, J = 8 / T, NT = G / T;
    typedef float Vec __attribute__((ext_vector_type(V)));
};

// C[v][c] = X[v][c] / outdeg(v) (0 for dangling v), over all n x W entries; the rows of
// zeros behind C and D.
template <int W>
__global__ __launch_bounds__(BLK) void ppr_contrib(PprArgs a, float *C) {
    const int64_t total = (int64_t)a.n * W;
    for (int64_t i = blockIdx.x * (int64_t)BLK + threadIdx.x; i < total; i += (int64_t)gridDim.x * BLK) {
        const int v = (int)(i / W);
        const int d = a.out_off[v + 1] - a.out_off[v];
        C[i] = d > 0 ? a.X[i] / (float)d : 0.f;
    }
    if (blockIdx.x == 0 && threadIdx.x < W) {
        C[total + threadIdx.x] = 0.f;
        a.D[total + threadIdx.x] = 0.f;
    }
}

// A block's sum in the lane's columns: the eight in-edges of the list (`len` long, at in_adj +
// beg) from offset e on, past its end the row of zeros.  Two lanes load four sources each
// (a.m bounds the array), quad permutes spread them, and the eight rows are gathered together.
template <int W, bool WIDE>
__device__ __forceinline__ typename PprLanes<W>::Vec ppr_block(const PprArgs &a, int beg, int len, int e) {
    using P = PprLanes<W>;
    typedef int Int4 __attribute__((ext_vector_type(4), aligned(4)));
    e += 4 * (lane_id() & 1);
    const int at = beg + (e < len ? e : 0);
    Int4 x;
    if (at + 4LL <= a.m) {
        x = *(const Int4 *)(a.in_adj + at);
    } else {
        x = a.n;
        for (int j = 0; j < 4; ++j)
            if (at + j < a.m) x[j] = a.in_adj[at + j];
    }
    typename P::Vec c[8];
    const uint32_t l = lane_id() % P::L * (4 * P::V);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int y = e + k % 4 < len ? x[k % 4] : a.n;
        const int u = P::L == 2 ? (k < 4 ? __builtin_amdgcn_mov_dpp(y, 0xA0, 0xF, 0xF, true)    // lanes 0, 0, 2, 2
                                         : __builtin_amdgcn_mov_dpp(y, 0xF5, 0xF, 0xF, true))   // lanes 1, 1, 3, 3
                                : (k < 4 ? __builtin_amdgcn_mov_dpp(y, 0x00, 0xF, 0xF, true)    // lane 0 of the quad
                                         : __builtin_amdgcn_mov_dpp(y, 0x55, 0xF, 0xF, true));  // lane 1
        const uint64_t off = WIDE ? (uint64_t)(uint32_t)u * (4 * W) + l : (uint64_t)((uint32_t)u * (4 * W) + l);
        c[k] = *(const typename P::Vec *)((const char *)a.C + off);
    }
    return ((c[0] + c[1]) + (c[2] + c[3])) + ((c[4] + c[5]) + (c[6] + c[7]));
}

// Sum of the lane's columns over a list of `len` in-edges, in one order for every width: the
// list is cut into blocks of eight edges, a block is summed as in ppr_block, block i is added
// to partial sum i mod 8 (each adds its blocks in order), and the partial sums are combined
// as ((s0 + s1) + (s2 + s3)) + ((s4 + s5) + (s6 + s7)).  Here a team sums one list: group g of
// its T sums blocks T i + g; the combination steps over partial sums on different groups are
// lane butterflies, the others adds inside the lane, and addition is commutative, so every
// width and every lane computes the same bits.
template <int W, bool WIDE>
__device__ __forceinline__ typename PprLanes<W>::Vec team_list(const PprArgs &a, int beg, int len, int steps) {
    using P = PprLanes<W>;
    const int g = lane_id() / P::L % P::T;
    typename P::Vec acc[P::J];
#pragma unroll
    for (int j = 0; j < P::J; ++j) acc[j] = 0.f;
    for (int i = 0; i < steps; i += P::J)
#pragma unroll
        for (int j = 0; j < P::J; ++j) {
            if (i + j >= steps) continue;
            acc[j] += ppr_block<W, WIDE>(a, beg, len, 8 * (P::T * (i + j) + g));
        }
    // partial sum g + T j is acc[j] of group g
    static_assert(P::T * P::J == 8, "eight partial sums");
#pragma unroll
    for (int b = 1; b < P::T; b *= 2)
#pragma unroll
        for (int j = 0; j < P::J; ++j)
#pragma unroll
            for (int i = 0; i < P::V; ++i) acc[j][i] += __shfl_xor(acc[j][i], P::L * b);
#pragma unroll
    for (int b = 1; b < P::J; b *= 2)
#pragma unroll
        for (int j = 0; j + b < P::J; j += 2 * b) acc[j] += acc[j + b];
    return acc[0];
}

// The same sums with a list per group, in `steps` blocks (the longest list's).
template <int W, bool WIDE>
__device__ __forceinline__ typename PprLanes<W>::Vec group_list(const PprArgs &a, int beg, int len, int steps) {
    typename PprLanes<W>::Vec acc[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[k] = 0.f;
    for (int i = 0; i < steps; i += 8)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (i + j >= steps) continue;
            acc[j] += ppr_block<W, WIDE>(a, beg, len, 8 * (i + j));
        }
    return ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
}

// The lane's columns of u from their sums, as ranks after the last iteration, as the
// contributions that the next one gathers before.  Idle columns are set too, to nothing that
// is looked at.
template <int W>
__device__ __forceinline__ void ppr_apply(const PprArgs &a, int u, typename PprLanes<W>::Vec s,
                                          const int (&src)[PprLanes<W>::V]) {
    using P = PprLanes<W>;
    const int d = a.out_off[u + 1] - a.out_off[u];
    typename P::Vec x;
#pragma unroll
    for (int i = 0; i < P::V; ++i) {
        const float v = (1.0f - a.t) * s[i];
        x[i] = u == src[i] ? a.t + v : v;
        if (!a.last) x[i] = d > 0 ? x[i] / (float)d : 0.f;
    }
    *(typename P::Vec *)(a.D + (int64_t)u * W + lane_id() % P::L * P::V) = x;
}

// One iteration.  WIDE: rows past 4 GiB.
template <int W, bool WIDE>
__global__ __launch_bounds__(BLK) void ppr_gather(PprArgs a) {
    using P = PprLanes<W>;
    const int lane = lane_id(), g = lane / P::L, l = lane % P::L, team = g / P::T;
    const int wave = (blockIdx.x * BLK + (int)threadIdx.x) / WAVE, nwaves = gridDim.x * BLK / WAVE;
    int src[P::V];
#pragma unroll
    for (int i = 0; i < P::V; ++i) src[i] = a.src[l * P::V + i];
    // pieces of long lists, one a team; the team that sums a list's last adds them all in
    // order, T loaded together
    for (int t0 = wave * P::NT; t0 < a.npart; t0 += nwaves * P::NT) {
        const int t = t0 + team;
        const ChunkRec r = a.tasks[min(t, a.npart - 1)];
        const int len = t < a.npart ? r.end - r.beg : 0;
        int steps = (len + 8 * P::T - 1) / (8 * P::T);
#pragma unroll
        for (int o = P::T * P::L; o < WAVE; o *= 2) steps = max(steps, __shfl_xor(steps, o));
        const auto s = team_list<W, WIDE>(a, r.beg, len, __builtin_amdgcn_readfirstlane(steps));
        if (len == 0) continue;
        int *big = a.big + 4 * r.pad;
        const int p0 = big[1], np = big[2];
        if (g % P::T == 0)
#pragma unroll
            for (int i = 0; i < P::V; ++i)
                __hip_atomic_store(&a.part[(int64_t)t * W + l * P::V + i], s[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // stored before it is counted
        const int first = team * P::T * P::L;
        int old = 0;
        if (lane == first) old = atomicAdd(&big[3], 1);
        if (__shfl(old, first) != np - 1) continue;
        typename P::Vec sum = 0.f;
        for (int p = 0; p < np; p += P::T) {
            const int64_t at = (int64_t)(p0 + min(p + g % P::T, np - 1)) * W + l * P::V;
            typename P::Vec x;
#pragma unroll
            for (int i = 0; i < P::V; ++i) x[i] = __hip_atomic_load(&a.part[at + i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int j = 0; j < P::T; ++j)
#pragma unroll
                for (int i = 0; i < P::V; ++i) {
                    const float y = __shfl(x[i], first + j * P::L + l);
                    if (p + j < np) sum[i] += y;
                }
        }
        if (lane == first) big[3] = 0;
        if (g % P::T == 0) ppr_apply<W>(a, r.v, sum, src);
    }
    // runs, G vertices at a time: a list per group, or, where that takes more steps, a list
    // per team, one after another
    for (int t = a.npart + wave; t < a.ntasks; t += nwaves) {
        const ChunkRec r = a.tasks[t];
        for (int u0 = r.v; u0 < r.v + r.pad; u0 += P::G) {
            const int u = u0 + g;
            const bool has = u < r.v + r.pad;
            const int b = has ? a.in_off[u] : 0, len = has ? a.in_off[u + 1] - b : 0;
            int longest = (len + 7) / 8, one = (len + 8 * P::T - 1) / (8 * P::T);
#pragma unroll
            for (int o = P::L; o < WAVE; o *= 2) {
                longest = max(longest, __shfl_xor(longest, o));
                one += __shfl_xor(one, o);
            }
            longest = __builtin_amdgcn_readfirstlane(longest);
            one = __builtin_amdgcn_readfirstlane(one);
            typename P::Vec s = 0.f;
            if (longest * P::NT <= one) {
                s = group_list<W, WIDE>(a, b, len, longest);
            } else {
                uint64_t some = wave_ballot(len > 0 && l == 0);  // bit g * L per list
                while (some) {
                    int at[P::NT];
#pragma unroll
                    for (int i = 0; i < P::NT; ++i) {
                        at[i] = some ? __ffsll((unsigned long long)some) - 1 : -1;
                        some &= some - 1;
                    }
                    const int mine = at[team], from = max(mine, 0);
                    int tb = __shfl(b, from), tl = __shfl(len, from);
                    if (mine < 0) tb = tl = 0;
                    int steps = 0;
#pragma unroll
                    for (int i = 0; i < P::NT; ++i)
                        steps = max(steps, at[i] < 0 ? 0 : (__builtin_amdgcn_readlane(len, at[i]) + 8 * P::T - 1) / (8 * P::T));
                    const auto sl = team_list<W, WIDE>(a, tb, tl, steps);
#pragma unroll
                    for (int i = 0; i < P::NT; ++i)
#pragma unroll
                        for (int c = 0; c < P::V; ++c) {
                            const float y = __shfl(sl[c], i * P::T * P::L + l);
                            if (at[i] / P::L == g && at[i] >= 0) s[c] = y;
                        }
                }
            }
            if (has) ppr_apply<W>(a, u, s, src);
        }
    }
}

// Rows of width w1 -> rows of width w2 (columns beyond w1 start at 0).
__global__ void ppr_repack(const float *X, int w1, float *Y, int w2, int n) {
    const int64_t total = (int64_t)n * w2;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t v = i / w2;
        const int c = (int)(i % w2);
        Y[i] = c < w1 ? X[v * w1 + c] : 0.f;
    }
}

// Column reset of the listed slots: x_0 = e_src.
__global__ void ppr_seed_cols(float *X, int n, int W, SeedList sl) {
    const int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, nt = (int64_t)gridDim.x * blockDim.x;
    for (int64_t u = tid; u < n; u += nt)
        for (int j = 0; j < sl.n; ++j) X[u * W + sl.slot[j]] = u == sl.src[j] ? 1.f : 0.f;
}

__global__ void ppr_set_src(int *src, SeedList sl, SlotList off) {
    const int i = threadIdx.x;
    if (i < off.n) src[off.slot[i]] = -1;
    __syncthreads();
    if (i < sl.n) src[sl.slot[i]] = sl.src[i];
}

// Rank columns of the listed slots -> their rows (64 vertices x W columns through LDS).
__global__ __launch_bounds__(BLK) void ppr_extract(const float *X, int W, float *rows, int n, SlotList sl) {
    __shared__ float tile[64][65];
    const int tv = (n + 63) / 64;
    for (int t = blockIdx.x; t < tv; t += gridDim.x) {
        const int v0 = t * 64;
        for (int i = threadIdx.x; i < 64 * W; i += BLK) {
            const int r = i / W, cc = i % W;
            tile[r][cc] = (v0 + r < n) ? X[(int64_t)(v0 + r) * W + cc] : 0.f;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < sl.n * 64; i += BLK) {
            const int j = i / 64, r = i % 64;
            if (v0 + r < n) rows[(int64_t)sl.slot[j] * n + v0 + r] = tile[r][sl.slot[j]];
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------- host side

void ppr_dev_free(PprDev &p) {
    free_dev(p.X[0]);
    free_dev(p.X[1]);
    free_dev(p.C);
    free_dev(p.part);
    free_dev(p.tasks);
    free_dev(p.big);
    free_dev(p.src);
    free_dev(p.rows);
    p = PprDev{};
}

// In-edge view for PageRank gathers: the CSR of a symmetric graph, else the CSC.
static bool ppr_view(const mg_graph *g, const int **off, const int **adj) {
    if (g->flags & MG_GRAPH_SYMMETRIC) {
        *off = g->row_off;
        *adj = g->col;
        return true;
    }
    if (g->col_off) {
        *off = g->col_off;
        *adj = g->row_idx;
        return true;
    }
    return false;
}

static int ppr_piece(const mg_graph *g) {
    return (int)std::clamp<int64_t>(g->m / PPR_PIECES / WAVE * WAVE, PPR_T_MIN, PPR_T_MAX);
}

int64_t ppr_dev_bytes(const mg_graph *g) {
    const int64_t n = g->n;
    const int T = ppr_piece(g);
    const int64_t tasks = g->m / T + n / PPR_RUN + 2 * (g->m / T) + 64;
    return 3 * 4LL * PPR_SLOTS * (n + 1) + 4LL * PPR_SLOTS * (g->m / T + 64) + (int64_t)sizeof(ChunkRec) * tasks +
           16LL * (g->m / T + 64) + 4LL * PPR_SLOTS + 4LL * PPR_SLOTS * n;
}

int ppr_dev_alloc(PprDev &p, mg_graph *g, hipStream_t st) {
    ppr_dev_free(p);
    const int *off = nullptr, *adj = nullptr;
    if (!ppr_view(g, &off, &adj))
        return set_error(MG_ERR_UNSUPPORTED, "personalized PageRank needs MG_GRAPH_SYMMETRIC or MG_GRAPH_BUILD_CSC");
    const int n = g->n;
    std::vector<int> h_off((size_t)n + 1);
    MG_HIP(copy_on(st, h_off.data(), off, 4 * ((size_t)n + 1), hipMemcpyDeviceToHost));
    const int T = ppr_piece(g);
    std::vector<ChunkRec> tasks, runs;
    std::vector<int> big;
    for (int v = 0; v < n;) {
        const int d = h_off[v + 1] - h_off[v];
        if (d > T) {
            big.insert(big.end(), {v, (int)tasks.size(), (d + T - 1) / T, 0});
            for (int b = h_off[v]; b < h_off[v + 1]; b += std::min(T, h_off[v + 1] - b))
                tasks.push_back(ChunkRec{v, b, b + std::min(T, h_off[v + 1] - b), (int)(big.size() / 4) - 1});
            ++v;
            continue;
        }
        int u = v, e = 0;
        while (u < n && u - v < PPR_RUN && h_off[u + 1] - h_off[u] <= T && e + (h_off[u + 1] - h_off[u]) <= T) {
            e += h_off[u + 1] - h_off[u];
            ++u;
        }
        runs.push_back(ChunkRec{v, 0, 0, u - v});
        v = u;
    }
    const int npart = (int)tasks.size();
    tasks.insert(tasks.end(), runs.begin(), runs.end());
    p.n = n;
    p.ntasks = (int)tasks.size();
    p.npart = npart;
    hipError_t e = hipSuccess;
    auto A = [&](void **q, size_t bytes) {
        if (e == hipSuccess) e = alloc_refused() ? hipErrorOutOfMemory : hipMalloc(q, bytes ? bytes : 16);
    };
    for (float **q : {&p.X[0], &p.X[1], &p.C}) A((void **)q, 4 * (size_t)PPR_SLOTS * (n + 1));
    A((void **)&p.part, 4 * (size_t)PPR_SLOTS * npart);
    A((void **)&p.tasks, sizeof(ChunkRec) * tasks.size());
    A((void **)&p.big, 4 * big.size());
    A((void **)&p.src, 4 * PPR_SLOTS);
    A((void **)&p.rows, 4 * (size_t)PPR_SLOTS * n);
    if (e == hipSuccess) e = copy_on(st, p.tasks, tasks.data(), sizeof(ChunkRec) * tasks.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess && !big.empty()) e = copy_on(st, p.big, big.data(), 4 * big.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        std::vector<int> none(PPR_SLOTS, -1);
        e = copy_on(st, p.src, none.data(), 4 * PPR_SLOTS, hipMemcpyHostToDevice);
    }
    if (e == hipSuccess) e = hipMemsetAsync(p.X[0], 0, 4 * (size_t)PPR_SLOTS * (n + 1), st);
    if (e == hipSuccess) e = hipMemsetAsync(p.X[1], 0, 4 * (size_t)PPR_SLOTS * (n + 1), st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) {
        ppr_dev_free(p);
        return set_error(MG_ERR_OOM, "personalized PageRank state allocation failed: %s", hipGetErrorString(e));
    }
    p.bytes = ppr_dev_bytes(g);
    return MG_OK;
}

// The row width for the slots in `live`.
static int ppr_width(uint64_t live) {
    const int need = live ? 64 - __builtin_clzll(live) : 1;
    return need <= 8 ? 8 : need <= 16 ? 16 : need <= 32 ? 32 : 64;
}

static PprArgs ppr_args(PprDev &p, mg_graph *g, float t) {
    PprArgs a{};
    ppr_view(g, &a.in_off, &a.in_adj);
    a.out_off = g->row_off;
    a.X = p.X[p.cur];
    a.part = p.part;
    a.tasks = p.tasks;
    a.big = p.big;
    a.src = p.src;
    a.m = g->m;
    a.n = p.n;
    a.npart = p.npart;
    a.ntasks = p.ntasks;
    a.t = t;
    return a;
}

int ppr_seed(PprDev &p, hipStream_t st, const SeedList &sl, const SlotList &retire) {
    uint64_t live = p.live;
    for (int i = 0; i < retire.n; ++i) live &= ~(1ull << retire.slot[i]);
    for (int i = 0; i < sl.n; ++i) live |= 1ull << sl.slot[i];
    const int w = ppr_width(live);
    if (w != p.width) {  // rows of the new width into the other buffer
        hipLaunchKernelGGL(ppr_repack, dim3(grid_blocks_cap((int64_t)p.n * w, BLK, 4 * MAX_GRID)), dim3(BLK), 0, st,
                           (const float *)p.X[p.cur], p.width, p.X[p.cur ^ 1], w, p.n);
        p.cur ^= 1;
        p.width = w;
    }
    p.live = live;
    if (sl.n > 0)
        hipLaunchKernelGGL(ppr_seed_cols, dim3(grid_blocks(p.n, BLK)), dim3(BLK), 0, st, p.X[p.cur], p.n, p.width, sl);
    hipLaunchKernelGGL(ppr_set_src, dim3(1), dim3(PPR_SLOTS), 0, st, p.src, sl, retire);
    MG_HIP(hipGetLastError());
    return MG_OK;
}

// A launch per iteration, contributions to contributions, the last one to ranks: through C
// and the spare rank buffer, and over the current ranks (needed by then for nothing) when the
// last contributions are in the spare one.
template <int W>
static int ppr_iterate_w(PprDev &p, mg_graph *g, hipStream_t st, float t, int iters) {
    if (iters <= 0 || p.live == 0) return MG_OK;
    PprArgs a = ppr_args(p, g, t);
    float *spare = p.X[p.cur ^ 1], *from = p.C;
    a.D = spare;
    hipLaunchKernelGGL(ppr_contrib<W>, dim3(grid_blocks_cap((int64_t)p.n * W, BLK, 4 * MAX_GRID)), dim3(BLK), 0, st, a, p.C);
    const int G = grid_blocks_cap((int64_t)p.ntasks * WAVE, BLK, 1 << 20);  // hardware hands them out as waves end
    const bool wide = ((uint64_t)p.n + 1) * W * 4 > UINT32_MAX;
    for (int i = 0; i < iters; ++i) {
        a.last = i == iters - 1;
        a.C = from;
        a.D = from == p.C ? spare : a.last ? p.X[p.cur] : p.C;
        if (wide) hipLaunchKernelGGL((ppr_gather<W, true>), dim3(G), dim3(BLK), 0, st, a);
        else hipLaunchKernelGGL((ppr_gather<W, false>), dim3(G), dim3(BLK), 0, st, a);
        from = a.D;
    }
    MG_HIP(hipGetLastError());
    if (from == spare) p.cur ^= 1;
    return MG_OK;
}

int ppr_iterate(PprDev &p, mg_graph *g, hipStream_t st, float t, int iters) {
    switch (p.width) {
    case 8: return ppr_iterate_w<8>(p, g, st, t, iters);
    case 16: return ppr_iterate_w<16>(p, g, st, t, iters);
    case 32: return ppr_iterate_w<32>(p, g, st, t, iters);
    default: return ppr_iterate_w<64>(p, g, st, t, iters);
    }
}

int ppr_extract_rows(PprDev &p, hipStream_t st, const SlotList &sl) {
    if (sl.n <= 0) return MG_OK;
    hipLaunchKernelGGL(ppr_extract, dim3(grid_blocks((int64_t)((p.n + 63) / 64) * BLK, BLK)), dim3(BLK), 0, st,
                       (const float *)p.X[p.cur], p.width, p.rows, p.n, sl);
    MG_HIP(hipGetLastError());
    return MG_OK;
}

int64_t ppr_dev_size(const PprDev *p) { return p->bytes; }

void ppr_release(mg_graph *g) {
    if (g->steps && g->steps->pdev) {
        ppr_dev_free(*g->steps->pdev);
        delete g->steps->pdev;
        g->steps->pdev = nullptr;
    }
}

int ppr_iters_of(const mg_options &o) { return o.ppr_iters > 0 ? o.ppr_iters : 20; }

}  // namespace mg

using namespace mg;

extern "C" int mg_ppr_batch(mg_graph *g, const int32_t *srcs, int32_t k, float *rank_out, const mg_options *opt,
                            mg_stats *stats) {
    CallTimer timer;
    mg_options o;
    int rc = begin_search(g, opt, &o);
    if (rc) return rc;
    std::lock_guard<std::mutex> lock(g->mu);
    if (k < 1 || k > PPR_SLOTS || !srcs)
        return set_error(MG_ERR_INVALID_ARG, "mg_ppr_batch: k must be in [1, %d] with a source array", PPR_SLOTS);
    if ((rc = check_batch_sources("mg_ppr_batch", g, srcs, k))) return rc;
    if (!(o.pr_teleport >= 0.f && o.pr_teleport <= 1.f))
        return set_error(MG_ERR_INVALID_ARG, "mg_ppr_batch: pr_teleport must be in [0, 1]");
    // the degree-ordered twin when the graph keeps one (sources renamed, rows mapped
    // back); its in-lists are in twin order, so the sums are the twin's, as for serving
    int32_t tsrc[PPR_SLOTS];
    mg_graph *sg = batch_graph(g, o, srcs, k, tsrc);
    if (sg != g) srcs = tsrc;
    PprDev *&p = sg->steps->pdev;
    if (!p) {
        p = new (std::nothrow) PprDev();
        if (!p) return set_error(MG_ERR_OOM, "host allocation failed");
        if ((rc = ppr_dev_alloc(*p, sg, g->stream))) {
            delete p;
            p = nullptr;
            return rc;
        }
    }
    SeedList sl{};
    SlotList retire{}, all{};
    retire.n = PPR_SLOTS;
    for (int s = 0; s < PPR_SLOTS; ++s) retire.slot[s] = s;
    sl.n = all.n = k;
    for (int s = 0; s < k; ++s) {
        sl.slot[s] = all.slot[s] = s;
        sl.src[s] = srcs[s];
    }
    const int iters = ppr_iters_of(o);
    MG_HIP(hipEventRecord(g->ev0, g->stream));
    if ((rc = ppr_seed(*p, g->stream, sl, retire))) return rc;
    if ((rc = ppr_iterate(*p, sg, g->stream, o.pr_teleport, iters))) return rc;
    if ((rc = ppr_extract_rows(*p, g->stream, all))) return rc;
    const float *result = p->rows;
    if (sg != g) {  // rows 0..k-1 back to the caller's ids, into the spare rank buffer
        float *spare = p->X[p->cur ^ 1];
        if ((rc = launch_unpermute_rows(sg->perm, (const int *)p->rows, g->n, k, (int *)spare, g->stream))) return rc;
        result = spare;
    }
    MG_HIP(hipEventRecord(g->ev1, g->stream));
    MG_HIP(hipEventSynchronize(g->ev1));
    float ms = 0;
    MG_HIP(hipEventElapsedTime(&ms, g->ev0, g->ev1));
    if (stats) {
        std::memset(stats, 0, sizeof *stats);
        stats->iterations = iters;
        stats->edges_traversed = (int64_t)k * g->m * iters;
        stats->vertices_reached = (int64_t)k * g->n;
        stats->device_ms = ms;
    }
    if ((rc = deliver(g, rank_out, result, 4 * (size_t)k * g->n, o.out_on_device))) return rc;
    if (stats) stats->host_ms = timer.ms();
    return MG_OK;
}
