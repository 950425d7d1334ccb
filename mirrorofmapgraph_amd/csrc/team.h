// Teams: the waves of a few workgroups of one launch that run narrow levels back to back.
//
// A level of a few thousand vertices is a chain of dependent memory accesses.  One
// workgroup (one CU) is bound by its own address rate there: a 2048^2 grid's BFS levels
// (about 1000 vertices, some 12 accesses to lines of their own each) took 17.5 us in one
// workgroup.  A team spreads a level over up to TEAM_WGS workgroups (64 waves) that meet
// between levels.  Its members are waves: each has its own part of the next frontier and
// posts for itself, so a level has no workgroup barrier and no shared counter.
//
// The workgroups of a team run on one XCD: they share its L2, so what one wave writes (L1
// is write-through) another reads there with a load that passes its L1 (agent scope).
// Measured on the MI355X: L2 hit 0.09 us, memory 0.38 us, returning atomic 0.28 us; a
// meeting of 16 workgroups on one XCD 0.56 us (post with a store, poll with loads) against
// 1.0 us when the post has to reach the other XCDs, and 2 us for 256 workgroups.
//
// A search asks for a team by pausing (Ctl::done = 2): its remaining queued steps do nothing
// and the host launches the team kernel, at once when the previous search's team is the
// guide (Ctl::team_step).  The kernel is no part of the steps: inlined into the level
// kernels it cost the searches that never use it 1 to 2%.
//
// Nothing waits for a workgroup that is not running: the first workgroup to arrive
// gathers others for at most TEAM_GATHER ticks, then closes the team; only workgroups
// that joined before take part, and they are resident until they leave.  A team may
// have any size from one workgroup.
#pragma once

#include "frontier.h"

namespace mg {

constexpr int TEAM_WGS = 16;                          // workgroups wanted
constexpr int TEAM_GRID = 16 * TEAM_WGS;               // workgroups launched: enough of them on one of 8 XCDs
constexpr int TEAM_SIZE = TEAM_WGS * (BLK / WAVE);    // members: their waves, one lane each in a meeting
static_assert(TEAM_SIZE <= WAVE, "a wave reads every member's post, one per lane");
constexpr int TEAM_SEG = 512;        // records a member queues per level
constexpr int TEAM_EDGES = 4;        // edges per record, a lane each
constexpr int TEAM_PIECE = WAVE / TEAM_EDGES;  // records a wave takes at a time
constexpr int TEAM_DEG = 1020;       // out-edges of a vertex a team queues (64 fit team_word's fields)
constexpr int TEAM_GATHER = 1000;    // ticks (100 MHz) the first member waits for others
constexpr int TEAM_CLOSED = 1 << 29;

// Records: 1..TEAM_EDGES consecutive edge slots of a frontier vertex, TEAM_SEG records
// per member and buffer.
constexpr size_t TEAM_RECS = 2 * (size_t)TEAM_SIZE * TEAM_SEG;
static_assert(TEAM_EDGES == 4, "two bits of a record");
__host__ __device__ constexpr uint64_t team_record(int v, int beg, int len) {
    return (uint64_t)(uint32_t)v | ((uint64_t)(uint32_t)beg << 31) | ((uint64_t)(len - 1) << 62);
}
__device__ __forceinline__ int rec_vertex(uint64_t r) { return (int)r & 0x7fffffff; }
__device__ __forceinline__ int rec_beg(uint64_t r) { return (int)(r >> 31) & 0x7fffffff; }
__device__ __forceinline__ int rec_len(uint64_t r) { return (int)(r >> 62) + 1; }

// What a member posts after a level (of its part of the next frontier): tag (the
// meeting's number, 11 bits), overflow, records, vertices, out-edges.  A member
// whose counts do not fit posts the overflow bit.
__host__ __device__ constexpr uint64_t team_word(int tag, bool over, int rec, int nf, int mf) {
    return ((uint64_t)(tag & 0x7ff) << 53) | ((uint64_t)over << 52) | ((uint64_t)rec << 36) | ((uint64_t)nf << 20) |
           (uint64_t)mf;
}
__device__ __forceinline__ int team_tag(uint64_t w) { return (int)(w >> 53); }
__device__ __forceinline__ bool team_over(uint64_t w) { return (w >> 52) & 1; }
__device__ __forceinline__ int team_rec(uint64_t w) { return (int)(w >> 36) & 0xffff; }
__device__ __forceinline__ int team_nf(uint64_t w) { return (int)(w >> 20) & 0xffff; }
__device__ __forceinline__ int team_mf(uint64_t w) { return (int)w & 0xfffff; }

struct TeamCtl {
    int leader, pad0[31];  // XCD of the team + 1 (0: none yet)
    int joined, pad1[31];
    int size;              // workgroups, once closed
    int hub, pad2[30];     // batches: a member overflowed at a vertex of more than TEAM_DEG edges
    uint64_t word[2][TEAM_SIZE];  // posts, by meeting parity
    int least[2][TEAM_SIZE];      // SSSP: a member's smallest waiting distance, by meeting parity
};

// The XCD this wave runs on (hardware register XCC_ID).
__device__ __forceinline__ int xcd_id() { return (int)__builtin_amdgcn_s_getreg(20 | (3 << 11)) & 15; }

// Before the launch that forms the team (one workgroup of at least 2 * TEAM_SIZE threads):
// nobody has joined, nothing is posted (meetings are numbered from 1).
template <int = 0>
__global__ void team_open(TeamCtl *t) {
    if (threadIdx.x < 2 * TEAM_SIZE) (&t->word[0][0])[threadIdx.x] = 0;
    if (threadIdx.x == 0) t->leader = t->joined = t->size = 0;
}

// Whole workgroup: joins the team of up to `wgs` (<= TEAM_WGS) workgroups.  False for
// workgroups that take no part; else this wave's number among the team's `size` waves (a
// workgroup's waves lie `size` / (BLK / WAVE) apart, so the first few members are on
// different CUs).
__device__ __forceinline__ bool team_join(TeamCtl *t, int wgs, int &rank, int &size) {
    __shared__ int s_rank, s_size;
    if (threadIdx.x == 0) {
        const int x = xcd_id() + 1;
        int r = wgs, n = 0;
        int lead = ld_dev(&t->leader);
        if (lead == 0) {
            lead = atomicCAS(&t->leader, 0, x);
            if (lead == 0) lead = x;
        }
        // (the load spares late workgroups the atomic)
        if (lead == x && ld_dev(&t->joined) < wgs) r = atomicAdd(&t->joined, 1);
        if (r == 0) {
            const long long t0 = wall_clock64();
            while (ld_dev(&t->joined) < wgs && wall_clock64() - t0 < TEAM_GATHER) __builtin_amdgcn_s_sleep(1);
            n = min(atomicOr(&t->joined, TEAM_CLOSED), wgs);
            __hip_atomic_store(&t->size, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else if (r < wgs) {
            // joined before the team closed: the first member is running and will close it
            while ((n = ld_dev(&t->size)) == 0) __builtin_amdgcn_s_sleep(1);
        }
        s_rank = r;
        s_size = n;
    }
    __syncthreads();
    if (s_rank >= s_size) return false;
    rank = __builtin_amdgcn_readfirstlane((int)threadIdx.x / WAVE * s_size + s_rank);
    size = __builtin_amdgcn_readfirstlane(s_size * (BLK / WAVE));
    return true;
}

__device__ __forceinline__ void team_set_hub(TeamCtl *t) {
    if (lane_id() == 0) __hip_atomic_store(&t->hub, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Whole wave: everything it wrote has reached the L2, then its post.
__device__ __forceinline__ void team_post(TeamCtl *t, int meeting, int rank, uint64_t word) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (lane_id() == 0)
        __hip_atomic_store(&t->word[meeting & 1][rank], word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Whole wave: waits until every member posted for the meeting; lane i < size gets
// member i's word, the others 0.  A post is kept until the meeting after the next, which
// no member reaches before all have read it.
__device__ __forceinline__ uint64_t team_meet(const TeamCtl *t, int meeting, int size) {
    const int lane = lane_id();
    uint64_t w = 0;
    for (;;) {
        if (lane < size)
            w = __hip_atomic_load(&t->word[meeting & 1][lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (!wave_ballot(lane < size && team_tag(w) != (meeting & 0x7ff))) break;
    }
    asm volatile("" ::: "memory");  // what the members wrote is read after this point
    return w;
}

// Inclusive sum over the lanes up to this one (DPP row shifts, then row ends carried).
__device__ __forceinline__ int wave_scan_add(int x) {
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, true);  // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, true);  // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, true);  // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, true);  // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // row_bcast:15 -> rows 1, 3
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // row_bcast:31 -> rows 2, 3
    return x;
}

// Sum over the wave, in every lane.
__device__ __forceinline__ int wave_total(int x) { return __builtin_amdgcn_readlane(wave_scan_add(x), WAVE - 1); }

// off[v] and off[v + 1] in one load.
struct __attribute__((packed, aligned(4))) IntPair {
    int a, b;
};
__device__ __forceinline__ IntPair ld_range(const int *off, int v) {
    return *reinterpret_cast<const IntPair *>(off + v);
}

// The words of a frontier bitmap, shared out over the team: calls fn(i, word) with K words
// of the wave read together (the whole wave calls it; word = 0 past the end).  The loads
// pass the L1, as other members may have written the words.
template <class Fn>
__device__ __forceinline__ void team_words(const uint32_t *bm, int nwords, int rank, int size, Fn fn) {
    constexpr int K = 4;
    for (int w0 = rank * WAVE + lane_id(); w0 - lane_id() < nwords; w0 += K * size * WAVE) {
        uint32_t word[K];
#pragma unroll
        for (int k = 0; k < K; ++k) word[k] = (uint32_t)ld_dev((const int *)bm + min(w0 + k * size * WAVE, nwords - 1));
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int i = w0 + k * size * WAVE;
            fn(i, i < nwords ? word[k] : 0u);
        }
    }
}

// The records of a meeting, as a wave sees them: lane i holds member i's count, and the
// end of its pieces (TEAM_PIECE records each) in the order of the members.
struct TeamIn {
    const uint64_t *recs;
    int have, end, pieces;
};
__device__ __forceinline__ TeamIn team_in(const uint64_t *recs, int meeting, uint64_t word) {
    TeamIn t;
    t.recs = recs + (size_t)(meeting & 1) * TEAM_SIZE * TEAM_SEG;
    t.have = team_rec(word);
    t.end = wave_scan_add((t.have + TEAM_PIECE - 1) / TEAM_PIECE);
    t.pieces = __builtin_amdgcn_readlane(t.end, WAVE - 1);
    return t;
}
// This lane's record of piece p < pieces (TEAM_EDGES lanes share one); `on` is cleared
// where the piece is shorter (the lane then gets a real record all the same).
__device__ __forceinline__ uint64_t team_fetch(const TeamIn &t, int p, bool &on) {
    const int s = __popcll(wave_ballot(t.end <= p));  // the member whose piece it is
    const int left = __builtin_amdgcn_readlane(t.end, s) - p;  // its pieces from p on
    const int have = __builtin_amdgcn_readlane(t.have, s);
    const int r = ((have + TEAM_PIECE - 1) / TEAM_PIECE - left) * TEAM_PIECE + lane_id() / TEAM_EDGES;
    on = on && r < have;
    return __hip_atomic_load(&t.recs[(size_t)s * TEAM_SEG + min(r, have - 1)], __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}

// A wave's place in a team.
struct TeamSeat {
    TeamCtl *ctl;
    uint64_t *recs;  // TEAM_RECS records
    int rank, size;
};

// A member's part of the next frontier.
struct TeamOut {
    uint64_t *recs;
    int nrec = 0, nf = 0, mf = 0;
    bool hub = false;  // a vertex of more than TEAM_DEG edges
    __device__ TeamOut(uint64_t *all, int meeting, int rank)
        : recs(all + ((size_t)(meeting & 1) * TEAM_SIZE + rank) * TEAM_SEG) {}
    // Whole wave: queues vertex v with edge slots o.a..o.b for every lane with `first`
    // (`firsts`, not empty).
    __device__ __forceinline__ void queue(bool first, uint64_t firsts, int v, IntPair o) {
        const int deg = first ? o.b - o.a : 0;
        if (wave_ballot(deg > TEAM_DEG)) hub = true;
        // records and edges, one scan for both
        const int mine = min(deg, TEAM_DEG), mrec = (mine + TEAM_EDGES - 1) / TEAM_EDGES;
        const int sum = wave_scan_add(mrec << 16 | mine);
        const int all = __builtin_amdgcn_readlane(sum, WAVE - 1);
        int at = nrec + (sum >> 16) - mrec;
        for (int e = 0; e < mine && at < TEAM_SEG; e += TEAM_EDGES, ++at)
            __hip_atomic_store(&recs[at], team_record(v, o.a + e, min(mine - e, TEAM_EDGES)), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
        nf += __popcll(firsts);
        nrec += all >> 16;
        mf += all & 0xffff;
    }
    __device__ __forceinline__ uint64_t word(int meeting) const {
        const bool o = hub || nrec > TEAM_SEG || nf > 0xffff || mf > 0xfffff;
        return o ? team_word(meeting, true, 0, 0, 0) : team_word(meeting, false, nrec, nf, mf);
    }
};

}  // namespace mg
