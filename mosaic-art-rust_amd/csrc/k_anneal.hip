// k_anneal.hip -- adjacency cost, swap deltas and simulated annealing
// (AdjacencyPenaltyCalculator::calculate_total_cost / calculate_swap_delta /
// calculate_penalty, src/adjacency.rs:63-214; MosaicOptimizer::optimize and
// optimize_greedy, src/optimizer.rs:41-198).
//
// Annealing keeps the reference's one-proposal-at-a-time semantics exactly
// while a workgroup evaluates 64 proposals a round:
//   * proposal `it` draws x1,y1,x2,y2,u from a counter RNG keyed by (seed,it),
//     so any proposal can be evaluated out of order;
//   * skipped proposals (same cell / empty cell) do not cool, and emptiness
//     never changes under swaps, so proposal j's temperature index is the
//     number of non-skipped proposals before it (a ballot prefix count) and
//     T comes from a table built by the sequential f32 recurrence T *= decay;
//   * a round commits the proposals before the first that may have been
//     evaluated on other values than the serial chain would have read; the
//     rest are evaluated again in the next round;
//   * the running cost is accumulated in proposal order (f32, as the
//     reference's `current_cost += delta`).
// Result: grid, costs and counts are bit-identical to the serial chain.
#include "mh_device.hpp"
#include "mh_kernels.hpp"

#include <type_traits>

namespace mh {

// -------------------------------------------------------------- helpers
template <typename G>
__device__ __forceinline__ int32_t gget(const G* g, int32_t i) {
    return (int32_t)g[i];
}
template <typename G>
__device__ __forceinline__ void gput(G* g, int32_t i, int32_t v) {
    g[i] = (G)v;
}

// A grid kept in HBM (annealing of grids too large for LDS).  Every access
// is an agent-scope atomic, so a read never sees a stale cache line of a
// cell another lane of the wave has just written.
struct HbmGrid {
    int32_t* p;
};
__device__ __forceinline__ int32_t gget(const HbmGrid* g, int32_t i) {
    return __hip_atomic_load((MH_GAS int32_t*)g->p + i, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void gput(HbmGrid* g, int32_t i, int32_t v) {
    __hip_atomic_store((MH_GAS int32_t*)g->p + i, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One adjacency term 1/(sim(a,b)+1) from a Lab table in memory or in LDS.
struct TermLab {
    const float4* lab4;
    __device__ __forceinline__ float operator()(int32_t a, int32_t b) const {
        return adj_term(gload4(lab4, a), gload4(lab4, b));
    }
};
struct TermLds {
    const float4* labs;
    __device__ __forceinline__ float operator()(int32_t a, int32_t b) const {
        return adj_term(labs[a], labs[b]);
    }
};

// calculate_swap_delta (src/adjacency.rs:133-214): neighbours of p1 (Up,
// Down, Left, Right, skipping p2), then of p2 (skipping p1), then the mutual
// term when adjacent.  Absent terms are added as +0.0: the sums start at +0
// and only grow, and x + (+0) == x bit for bit, so this equals skipping them.
// Bound by latency: all ten cells are read at once, then their Labs (a neighbour
// outside reads its own cell, an empty one material 0's Lab).
__device__ float swap_delta_dev(const int32_t* grid, int32_t gw, int32_t gh, const float4* lab4,
                                int32_t x1, int32_t y1, int32_t x2, int32_t y2) {
    const int32_t p1 = y1 * gw + x1, p2 = y2 * gw + x2;
    const int32_t m1 = gget(grid, p1), m2 = gget(grid, p2);
    int32_t a[8];
    bool adjacent = false;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int32_t x = i < 4 ? x1 : x2, y = i < 4 ? y1 : y2, p = i < 4 ? p1 : p2;
        const int k = i & 3;
        const bool in = k == 0 ? y > 0 : k == 1 ? y < gh - 1 : k == 2 ? x > 0 : x < gw - 1;
        const int32_t q = k == 0 ? p - gw : k == 1 ? p + gw : k == 2 ? p - 1 : p + 1;
        const bool self = in && q == (i < 4 ? p2 : p1);  // the swap partner
        adjacent = adjacent || self;
        const int32_t v = gget(grid, in ? q : p);
        a[i] = in && !self ? v : kEmpty;
    }
    if (m1 == kEmpty || m2 == kEmpty || m1 == m2) return 0.0f;
    const float4 l1 = gload4(lab4, m1), l2 = gload4(lab4, m2);
    float4 la[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) la[i] = gload4(lab4, max(a[i], 0));
    float old_cost = 0.0f, new_cost = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float t1 = adj_term(l1, la[i]), t2 = adj_term(l2, la[i]);
        const bool there = a[i] != kEmpty;
        old_cost += there ? (i < 4 ? t1 : t2) : 0.0f;
        new_cost += there ? (i < 4 ? t2 : t1) : 0.0f;
    }
    if (adjacent) {
        const float t = adj_term(l1, l2);
        old_cost += t;
        new_cost += t;
    }
    return new_cost - old_cost;
}

// ------------------------------------------------------------ ordered sums
// s + t[0] + t[1] + ... in this order, each addition rounded to f32.  One
// dependent addition after another takes 10 ns (its read included), but most
// results are known without: while the sum s stays in one binade it is a
// whole number of the binade's ulps, and adding t adds t rounded to a whole
// number of ulps, whatever s is -- unless t lies half way between two, when
// the sum's last bit decides.  Whole numbers add in any order.
struct Ulps {
    uint32_t bits;
    // s in the normal range, its ulp and 1 / ulp too; else one by one
    __device__ __forceinline__ bool valid() const { return (bits >> 23) >= 23 && (bits >> 23) < 250; }
    __device__ __forceinline__ float per_unit() const {  // 1 / ulp(s)
        return __uint_as_float((277u - (bits >> 23)) << 23);
    }
    __device__ __forceinline__ int32_t count() const {
        return (int32_t)((bits & 0x7fffffu) | 0x800000u);
    }
    // the float of m ulps, 2^23 <= m < 2^24
    __device__ __forceinline__ float value(int32_t m) const {
        return __uint_as_float((bits & 0xff800000u) | ((uint32_t)m & 0x7fffffu));
    }
};
// f = t / ulp (exact but for what is rounded to 0 anyway): whether its whole
// number is certain, and small enough that 256 of them fit 32 bits.
__device__ __forceinline__ bool certain(float f, float r) {
    return __builtin_fabsf(f) <= 4194304.0f && __builtin_fabsf(f - r) != 0.5f;
}
// Inclusive sums over the lanes: within rows of 16, then over the rows.
__device__ __forceinline__ int32_t wave_scan_add(int32_t m) {
    m += __builtin_amdgcn_update_dpp(0, m, 0x111, 0xF, 0xF, false);
    m += __builtin_amdgcn_update_dpp(0, m, 0x112, 0xF, 0xF, false);
    m += __builtin_amdgcn_update_dpp(0, m, 0x114, 0xF, 0xF, false);
    m += __builtin_amdgcn_update_dpp(0, m, 0x118, 0xF, 0xF, false);
    m += __builtin_amdgcn_update_dpp(0, m, 0x142, 0xA, 0xF, false);
    m += __builtin_amdgcn_update_dpp(0, m, 0x143, 0xC, 0xF, false);
    return m;
}

// Inclusive minima over the lanes, the same way (no NaN).
__device__ __forceinline__ float wave_scan_min(float v) {
#define MH_MIN_STEP(CTRL, ROWS)                                                                    \
    v = __builtin_fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(                             \
                               __float_as_int(v), __float_as_int(v), CTRL, ROWS, 0xF, false)))
    MH_MIN_STEP(0x111, 0xF);
    MH_MIN_STEP(0x112, 0xF);
    MH_MIN_STEP(0x114, 0xF);
    MH_MIN_STEP(0x118, 0xF);
    MH_MIN_STEP(0x142, 0xA);
    MH_MIN_STEP(0x143, 0xC);
#undef MH_MIN_STEP
    return v;
}

// Adds the 64 lanes' t to s in lane order; returns each lane's sum (lane 63's
// is the total, which s becomes).  A lane that is half way, or whose sum
// leaves the inside of the binade, is added as it is, after the lanes below.
__device__ __forceinline__ float add_lanes(float& s, float t, int lane) {
    float c = s;
    int done = -1;  // the last lane added
    for (;;) {
        const Ulps U{__float_as_uint(s)};
        int32_t m = 0;
        bool stop = true;
        if (U.valid()) {
            const float f = t * U.per_unit(), r = __builtin_rintf(f);
            const bool sure = certain(f, r);
            m = U.count() + wave_scan_add(sure ? (int32_t)r : 0);
            stop = !sure || m <= 0x800000 || m >= 0x1000000;
        }
        // (a lane that adds nothing changes nothing)
        const uint64_t at = wave_ballot(stop && t != 0.0f);
        if (!at) {
            if (lane > done) c = wave_ballot(t != 0.0f) ? U.value(m) : s;
            s = readlane_f(c, 63);
            return c;
        }
        const int l = __ffsll((unsigned long long)at) - 1;
        const float v = lane > done && lane < l && U.valid() ? U.value(m) : s;
        if (lane > done) c = v;
        if (l > 0) s = readlane_f(c, l - 1);
        s = s + readlane_f(t, l);
        if (lane >= l) c = s;
        if (lane <= l) t = 0.0f;
        done = l;
    }
}

// The total alone, for sums that start at 0, in whose first binades many terms
// are half way: at once, or one by one (8 cycles each).
__device__ __forceinline__ float sum_lanes(float s, float t) {
    const Ulps U{__float_as_uint(s)};
    if (U.valid()) {
        const float f = t * U.per_unit(), r = __builtin_rintf(f);
        if (!wave_ballot(!certain(f, r))) {
            const uint32_t m = (uint32_t)U.count() + wave_sum_u32((uint32_t)r);
            if (m < 0x1000000u) return U.value((int32_t)m);
        }
    }
#pragma unroll
    for (int i = 0; i < 64; ++i) s = s + readlane_f(t, i);
    return s;
}

// calculate_total_cost (src/adjacency.rs:91-130) by one workgroup of
// kAnnealThreads, in the reference's order (raster, right before down).  An
// absent term is added as +0.0: the running sum starts at +0 and only grows,
// and x + (+0) == x bit for bit, so this equals skipping it.
//
// A wave takes 128 cells, two a lane, and rounds their 256 terms to the
// sum's ulps; the waves' sums are added while they are certain and stay in
// the binade.  Otherwise the wave whose turn it is adds its terms 64 at a time
// or one by one, and the waves after it round theirs again.  (Some 10 to 20 times a
// run: mostly the binades of the first few hundred terms.)  24,000 cells:
// 50 us, 450 us one by one.  lds: kCostWords words, 16-byte aligned.
// The result is returned to every wave.
constexpr int32_t kCostWaves = 12, kCostWords = 256 + 2 * kCostWaves + 4;
constexpr int32_t kAnnealThreads = 64 * kCostWaves;

template <typename G, typename TS>
__device__ float total_cost_block(const G* grid, int32_t gw, int32_t gh, const TS& T, uint32_t* lds) {
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    float* const strip = reinterpret_cast<float*>(lds);
    uint32_t* const sums = lds + 256;                // two buffers of kCostWaves
    uint32_t* const total = sums + 2 * kCostWaves;
    const int32_t cells = gw * gh;
    constexpr uint32_t kUnsure = 0xffffffffu;
    float s = 0.0f;
    int buffer = 0;
    constexpr int32_t kStep = 128 * kCostWaves;
    const int32_t step_x = kStep % gw, step_y = kStep / gw;
    const int32_t c0 = w * 128 + 2 * lane;
    int32_t x0 = c0 % gw, y0 = c0 / gw;
    for (int32_t base = 0; base < cells; base += kStep) {
        const int32_t c = base + c0;
        int32_t x = x0, y = y0;
        x0 += step_x;
        y0 += step_y + (x0 >= gw ? 1 : 0);
        x0 -= x0 >= gw ? gw : 0;
        float t[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int32_t p = c + i;
            const int32_t m = p < cells ? gget(grid, p) : kEmpty;
            if (m != kEmpty) {
                const int32_t r = x < gw - 1 ? gget(grid, p + 1) : kEmpty;
                const int32_t d = y < gh - 1 ? gget(grid, p + gw) : kEmpty;
                if (r != kEmpty) t[2 * i] = T(m, r);
                if (d != kEmpty) t[2 * i + 1] = T(m, d);
            }
            ++x;
            if (x == gw) {
                x = 0;
                ++y;
            }
        }
        for (int32_t done = 0; done < kCostWaves;) {
            const Ulps U{__float_as_uint(s)};
            bool sure = true;
            uint32_t sum = 0;
            const float inv = U.per_unit();
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float f = t[i] * inv, r = __builtin_rintf(f);
                sure = sure && certain(f, r);
                sum += (uint32_t)r;
            }
            if (!U.valid()) {  // sure of nothing but zeros
                sure = t[0] == 0.0f && t[1] == 0.0f && t[2] == 0.0f && t[3] == 0.0f;
                sum = 0;
            }
            sum = wave_ballot(!sure) ? kUnsure : wave_sum_u32(sum);
            if (lane == 0) sums[buffer + w] = sum;
            __syncthreads();
            int32_t m = U.count();
            bool going = true;
#pragma unroll
            for (int k = 0; k < kCostWaves; ++k) {
                const uint32_t v = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)sums[buffer + k]);
                going = going && (k < done || (v != kUnsure && (uint32_t)m + v < 0x1000000u));
                if (going && k >= done) {
                    m += (int32_t)v;
                    done = k + 1;
                }
            }
            buffer = kCostWaves - buffer;
            s = U.value(m);
            if (done == kCostWaves) break;
            if (w == done) {
                reinterpret_cast<float4*>(strip)[lane] = make_float4(t[0], t[1], t[2], t[3]);
                asm volatile("" ::: "memory");  // (one wave's LDS operations are done in order)
#pragma unroll 1
                for (int i = 0; i < 4; ++i) s = sum_lanes(s, strip[64 * i + lane]);
                if (lane == 0) *total = __float_as_uint(s);
            }
            __syncthreads();
            s = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int32_t)*total));
            ++done;
        }
    }
    return s;
}

// ---------------------------------------------------------- annealing
// What bounds it is the latency of a round, and how many proposals a round
// commits.  Small grids begin in whole blocks (follow_blocks, below), which commit
// more; what follows is the general form.  A round runs on twelve waves of one workgroup in two phases, with a
// barrier after each (s: the first proposal of the round; lane l of the slot
// waves and the judge: proposal s + l):
//   * terms: slot wave w makes the adjacency terms of one of the eight
//     neighbour cells with the swap's two materials.  The judge takes in the
//     proposals, and swaps those it expects to be accepted.
//   * decisions: the judge adds a swap's terms in the reference's order and
//     decides it.  The slot waves read the next round's cells and Labs, from
//     the grid as it is expected to be.
// If a decision was not the expected one, the judge puts the grid right and
// the next round begins with its reads once more (a third phase).  Meanwhile
// two waves draw later proposals and one adds the deltas to the running cost.
//
// A round's prefix that can be committed, `first`, is found in one of two
// ways, by which is longer for the share p of proposals that are accepted:
//   * expecting all of them to be accepted (the usual case: annealing starts
//     hot): in the first phase every lane stamps its two cells (the lowest
//     lane wins).  A neighbour stamped by a lower lane k is taken to be what
//     k's swap moves there: k's other material, whose Lab is in LDS.  A lane
//     one of whose own cells is stamped by a lower lane ends the prefix, and
//     so does one with a neighbour taken from a lane that is then rejected.
//     The lanes before `first` have 2 cells each, all different, so who wrote
//     a cell last, and what k held, is as assumed.  A lane ends it with a
//     probability of (4 + 16 (1 - p)) / cells for each lane below it.
//   * expecting none: every lane reads the cells as they are, accepted lanes
//     stamp theirs, and a lane with a lower lane's stamp on any of its ten
//     cells ends the prefix: 20 p / cells.
// The second is better for p < 5/9, over the last eight rounds or so: a round of a
// small grid decides a few proposals, too few to tell by (5,000 on 300 cells, 39%
// accepted: 1,065 -> 977 us).
//
// Measured against one wave that gathered its terms from a matrix of all pairs
// and added the initial cost one term after another: 1,000 proposals on 20 x
// 15 cells 332 -> 112 us (200 rounds -> 97; in 17 blocks 44 us), 2,000 on 80 x 60
// 340 -> 84 (100 -> 54), 2,000 on 206 x 116 600 -> 120, 20,000 on 200 x 120 1,650
// -> 488.  A round takes 1.0 us for 3.3 (1.5 with the reads as a
// phase of their own, 1.15 with two neighbours to each of four slot waves):
// 1,450 cycles of terms (the judge's taking in), 1,150 of decisions.
constexpr int kMarkWave = 9;  // in whole blocks; wave 10 draws
constexpr int kSlotWaves = 8, kJudgeWave = 8, kDraw1Wave = 9, kDraw2Wave = 10, kCostWave = 11;
static_assert(kAnnealThreads == 64 * (kCostWave + 1), "one wave a role");

// Stamps, tag << 7 | (63 - lane) << 1 | cell (0: the first of the swap): one
// word per cell, or for grids of more cells kHashStamps words that cells
// share (p mod kHashStamps).  A shared word can make a lane see a stamp that
// is not its cell's: that only ends the prefix early, or is found out by
// comparing the cells (substituted neighbours).  The words double as the
// initial cost's.
constexpr int32_t kHashStamps = 16384;
// A run that begins in whole blocks (follow_blocks) has two tables of 8 bytes a
// cell in the same place.
__host__ __device__ __forceinline__ int32_t stamp_words(int32_t cells, bool blocks) {
    if (cells > kHashStamps) return kHashStamps;
    const int32_t w = blocks ? 4 * cells : (cells + 3) & ~3;
    return w < kCostWords ? kCostWords : w;
}
constexpr uint32_t kTagEnd = (1u << 25) - 2u;  // (a round takes at most two)
// Proposal draws, made ahead into a ring of three words a slot: x1 | y1 << 16,
// x2 | y2 << 16, u (both sides are below 2^16: a grid in LDS is far smaller,
// and the HBM variant requires it).
constexpr int32_t kRing = 256;

// LDS in words, behind the stamps: Labs of the swaps' materials (64 of the
// first, 64 of the second), the terms (4 pairs of waves x 64 x {m1 with a, m2
// with a, m1 with b, m2 with b} for the pair's neighbours a, b), the lanes that
// the neighbours were taken from, the mutual terms, a round's accepted deltas,
// the ring, control words, the grid, the library's Labs (where they fit).
constexpr int32_t kLabWords = 2 * 64 * 4, kTermWords = kSlotWaves * 64 * 2,
                  kFromWords = kSlotWaves * 64, kMutualWords = 64, kPackWords = 2 * 64, kCtrlWords = 8;
constexpr int32_t kFixedWords =
    kLabWords + kTermWords + kFromWords + kMutualWords + kPackWords + 3 * kRing + kCtrlWords;
__host__ __device__ __forceinline__ int32_t grid_words(int32_t cells, int32_t kind) {
    return kind == kAnnealHbm ? 0 : (kind == kAnnealNarrow ? (cells + 7) / 8 * 4 : (cells + 3) & ~3);
}

// The control words: what a round leaves for the next, then a run's results.
enum { kCtrlRound = 0, kCtrlCost = 2, kCtrlBest = 3, kCtrlImproved = 4 };
__device__ __forceinline__ uint32_t pack_round(int32_t advance, bool hopeful, bool reread,
                                               int32_t accepted) {
    return (uint32_t)advance | (hopeful ? 128u : 0u) | (reread ? 256u : 0u) | (uint32_t)accepted << 9;
}

constexpr uint32_t kNoLane = 255u;

// How far a run has come.
struct Progress {
    int64_t s = 0, accepted = 0, evaluated = 0, rounds = 0;
};

template <typename G>
struct AnnealShared {
    uint32_t* stamp;
    float4* lab_m;     // [2][64]
    float4* terms;     // [kSlotWaves / 2][64]
    uint32_t* from;    // [kSlotWaves][64], kNoLane: none
    float* mutual;     // [64]
    float* pack;       // [2][64], the rounds use the first
    uint32_t *ring_xy1, *ring_xy2;
    float* ring_u;
    uint32_t* ctrl;
    const float4* labs;  // nullptr: read from the job's table in memory
    bool hashed;
    __device__ __forceinline__ int32_t at(int32_t p) const {
        return hashed ? p & (kHashStamps - 1) : p;
    }
};

// End of a phase: this wave's LDS operations are complete, then all waves
// meet.  (__syncthreads would also wait for loads in flight: the temperatures,
// which are requested a phase before their use.)
__device__ __forceinline__ void phase_end() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// How the waves follow the run, alike in each: the round's first proposal,
// the tag of its stamps, how its prefix is found, whether its reads must be
// repeated, and how many deltas the last round left.
struct Rounds {
    int64_t s;
    uint32_t tag = 1;
    bool hopeful = true, reread = false;
    int32_t pending = 0;

    // The last round's outcome.
    __device__ __forceinline__ void next(uint32_t ctrl) {
        const uint32_t v = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)ctrl);
        s += v & 127u;
        hopeful = (v & 128u) != 0u;
        reread = (v & 256u) != 0u;
        pending = (int32_t)(v >> 9);
    }
    // Before a round's terms; read: what the slot waves do to repeat the
    // reads, load: what a wave has to take in again then.  (Stamps of an old round look like this round's once the tags
    // wrap, so the stamps are cleared then.)
    template <typename G, typename Read, typename Load>
    __device__ __forceinline__ void begin(const AnnealShared<G>& S, int32_t words, int tid,
                                          Read&& read, Load&& load) {
        if (tag >= kTagEnd) {
            phase_end();
            for (int32_t i = tid; i < words; i += kAnnealThreads) S.stamp[i] = 0u;
            tag = 0;
            reread = true;
            phase_end();
        }
        if (reread) {
            ++tag;
            read();
            phase_end();
            load();
        }
    }
};
struct Nothing {
    __device__ __forceinline__ void operator()() const {}
};

// Where a slot wave's swap and its neighbour are (wave w & 3: Up, Down, Left,
// Right; w >> 2: of the swap's first, second cell).
struct Place {
    int32_t p1, p2, q;
    bool in, self;  // inside the grid; the swap's other cell
    bool active;
};

template <typename G>
__device__ __forceinline__ Place place_of(const AnnealJob& job, const AnnealShared<G>& S, int w,
                                          int64_t it) {
    const int32_t gw = job.grid_w;
    const bool vertical = !(w & 2), second = w >= 4, onward = w & 1;
    const int32_t step = vertical ? gw : 1, last = (vertical ? job.grid_h : gw) - 1;
    const uint32_t slot = (uint32_t)it & (kRing - 1);
    const uint32_t xy1 = S.ring_xy1[slot], xy2 = S.ring_xy2[slot];
    Place p;
    p.p1 = (int32_t)(xy1 >> 16) * gw + (int32_t)(xy1 & 0xffffu);
    p.p2 = (int32_t)(xy2 >> 16) * gw + (int32_t)(xy2 & 0xffffu);
    const int32_t centre = second ? p.p2 : p.p1, partner = second ? p.p1 : p.p2;
    const uint32_t xy = second ? xy2 : xy1;
    const int32_t along = (int32_t)(vertical ? xy >> 16 : xy & 0xffffu);
    p.in = along != (onward ? last : 0);
    // a neighbour outside the grid reads its own cell, always in bounds
    p.q = p.in ? centre + (onward ? step : -step) : centre;
    p.self = p.q == partner;  // (an outside one only where the proposal is skipped)
    p.active = it < job.max_iter && p.p1 != p.p2;
    return p;
}

// What a slot wave's reads bring: the neighbour's Lab, whether it counts, and
// whether the proposal does.
struct Reads {
    float4 lab;
    bool ok, skip;
};

template <typename G>
__device__ __forceinline__ Reads read_swap(const AnnealJob& job, const AnnealShared<G>& S, G* grid,
                                           int w, int lane, const Place& p, const Rounds& R) {
    const int32_t m1 = gget(grid, p.p1), m2 = gget(grid, p.p2), a = gget(grid, p.q);
    Reads r;
    r.skip = !p.active || m1 == kEmpty || m2 == kEmpty;
    r.ok = p.in && !p.self && a != kEmpty;
    // waves 0 and 4 read the swap's materials' Labs too
    const bool own = (w & 3) == 0;
    float4 lm = make_float4(0, 0, 0, 0);
    r.lab = lm;
    if (job.n > 0) {
        const int32_t i = max(a, 0), k = max(w == 0 ? m1 : m2, 0);
        if (S.labs) {
            r.lab = S.labs[i];
            if (own) lm = S.labs[k];
        } else {
            r.lab = gload4(job.lab4, i);
            if (own) lm = gload4(job.lab4, k);
        }
    }
    if (w == 2 && R.hopeful && !r.skip) {
        const uint32_t mine = (R.tag << 7) | ((uint32_t)(63 - lane) << 1);
        atomicMax(&S.stamp[S.at(p.p1)], mine);
        atomicMax(&S.stamp[S.at(p.p2)], mine | 1u);
    }
    if (own) S.lab_m[w * 16 + lane] = lm;
    return r;
}

// How many of the round's proposals are not blocked by a lower lane's stamp
// on one of their own cells (v1, v2: those cells' stamps), at most the rest of
// the run.
__device__ __forceinline__ int32_t expected_prefix(uint32_t v1, uint32_t v2, uint32_t mine, bool skip,
                                                   int64_t remain) {
    const bool taken = !skip && ((v1 >> 1) != (mine >> 1) || (v2 >> 1) != (mine >> 1));
    const uint64_t t = wave_ballot(taken);
    const int32_t first = t ? __ffsll((unsigned long long)t) - 1 : 64;
    return (int64_t)first < remain ? first : (int32_t)remain;
}

template <typename G>
__device__ __forceinline__ void slot_wave(const AnnealJob& job, const AnnealShared<G>& S, G* grid,
                                          int w, int lane, int32_t words,
                                          const Progress& P) {
    Rounds R;
    R.s = P.s;
    R.hopeful = !job.greedy;
    const int64_t max_iter = job.max_iter;
    Place p = place_of(job, S, w, P.s + lane);
    Reads r = read_swap(job, S, grid, w, lane, p, R);
    phase_end();
    for (;;) {
        // ---- terms
        const uint32_t outcome = S.ctrl[kCtrlRound];
        float4 l1, l2;
        uint32_t va, v1, v2;
        // (with the outcome in flight: it is nearly always the expected one)
        auto load = [&]() __attribute__((always_inline)) {
            va = S.stamp[S.at(p.q)];
            l1 = S.lab_m[lane];
            l2 = S.lab_m[64 + lane];
            v1 = S.stamp[S.at(p.p1)];
            v2 = S.stamp[S.at(p.p2)];
        };
        load();
        R.next(outcome);
        if (R.s >= max_iter) return;
        R.begin(
            S, words, w * 64 + lane,
            [&]() __attribute__((always_inline)) {
                p = place_of(job, S, w, R.s + lane);
                r = read_swap(job, S, grid, w, lane, p, R);
            },
            load);
        const uint32_t mine = (R.tag << 7) | ((uint32_t)(63 - lane) << 1);
        float4 la = r.lab;
        if (R.hopeful) {
            // stamped in this round by a lower lane: above this lane's stamps
            bool sub = va > (mine | 1u);
            uint32_t from = kNoLane;
            if (wave_ballot(sub)) {
                const uint32_t k = 63u - ((va >> 1) & 63u);
                bool first_cell = !(va & 1u);  // which of k's cells
                if (S.hashed) {
                    const uint32_t ks = (uint32_t)(R.s + k) & (kRing - 1);
                    const uint32_t k1 = S.ring_xy1[ks], k2 = S.ring_xy2[ks];
                    first_cell = (int32_t)(k1 >> 16) * job.grid_w + (int32_t)(k1 & 0xffffu) == p.q;
                    sub = sub && (first_cell || (int32_t)(k2 >> 16) * job.grid_w +
                                                        (int32_t)(k2 & 0xffffu) == p.q);
                }
                // k's first cell gets its second material, and the reverse
                const float4 other = S.lab_m[(first_cell ? 64u : 0u) + k];
                la = make_float4(sub ? other.x : la.x, sub ? other.y : la.y, sub ? other.z : la.z, 0.0f);
                from = sub ? k : kNoLane;
            }
            S.from[w * 64 + lane] = from;
        }
        const float t1 = adj_term(l1, la), t2 = adj_term(l2, la);
        reinterpret_cast<float2*>(S.terms)[((w >> 1) * 64 + lane) * 2 + (w & 1)] =
            make_float2(r.ok ? t1 : 0.0f, r.ok ? t2 : 0.0f);
        // the partner as a neighbour of the first cell: the mutual term
        if (w < 4 && p.self) S.mutual[lane] = t1;
        phase_end();
        // ---- decisions
        if (R.hopeful) {
            // the next round's proposals, if all goes as expected
            const int32_t first = expected_prefix(v1, v2, mine, r.skip, max_iter - R.s);
            p = place_of(job, S, w, R.s + first + lane);
            ++R.tag;
            r = read_swap(job, S, grid, w, lane, p, R);
        }
        phase_end();
    }
}

// What a swap adds to the cost, from its terms in the reference's order.
template <typename G>
__device__ __forceinline__ float added_terms(const AnnealShared<G>& S, int lane, bool adjacent) {
    const float4 t0 = S.terms[lane], t1 = S.terms[64 + lane], t2 = S.terms[128 + lane],
                 t3 = S.terms[192 + lane];
    // the first cell's neighbours: old with m1, new with m2; the second's the reverse
    float old_cost = t0.x, new_cost = t0.y;
    old_cost += t0.z;
    new_cost += t0.w;
    old_cost += t1.x;
    new_cost += t1.y;
    old_cost += t1.z;
    new_cost += t1.w;
    old_cost += t2.y;
    new_cost += t2.x;
    old_cost += t2.w;
    new_cost += t2.z;
    old_cost += t3.y;
    new_cost += t3.x;
    old_cost += t3.w;
    new_cost += t3.z;
    if (adjacent) {
        const float t = S.mutual[lane];
        old_cost += t;
        new_cost += t;
    }
    return new_cost - old_cost;
}

// Metropolis test u < exp(x), x = -delta/T (src/optimizer.rs:77-84).  An
// estimate from the hardware reciprocal and exp2 is within 2^-15 of exp(x),
// relative, down to 2^-126 (below, it may be 0, and u is either 0 or at least
// 2^-24), so it decides alone unless u lies within 2^-10 of it (or it is 0 or
// not finite); those lanes compute x and exp exactly.
__device__ __forceinline__ bool accepts(const AnnealJob& job, float delta, float temp, float u) {
    if (delta < 0.0f) return true;
    if (job.greedy) return false;
    const float e =
        __builtin_amdgcn_exp2f(-delta * __builtin_amdgcn_rcpf(temp) * 1.44269504f);
    if (__builtin_fabsf(u - e) > e * (1.0f / 1024.0f)) return u < e;
    return u < exp_f32(-delta / temp);
}

// kHbm: the grid's swaps are complete at agent scope before other waves read
// it (the barriers order the waves).
template <typename G, bool kHbm>
__device__ __forceinline__ void judge_wave(const AnnealJob& job, const AnnealShared<G>& S, G* grid,
                                           int lane, int32_t words, const Progress& P,
                                           AnnealOut* out) {
    Rounds R;
    R.s = P.s;
    R.hopeful = !job.greedy;
    const int32_t gw = job.grid_w, gh = job.grid_h;
    const int64_t max_iter = job.max_iter;
    int64_t kbase = P.evaluated, accepted = P.accepted, evaluated = P.evaluated, rounds = P.rounds;
    int32_t lean = 0;  // accepted shares above 5/9, decaying
    // the last round's, for the traces
    const bool traced = job.trace_delta || job.trace_accept;
    float delta = 0.0f;
    int64_t it = P.s + lane;
    bool acc = false, skip = true;
    int32_t first = 0;
    // the round's proposals (the next round's are taken in ahead)
    uint32_t xy1, xy2;
    float u;
    auto take = [&](int64_t from) __attribute__((always_inline)) {
        const uint32_t slot = (uint32_t)(from + lane) & (kRing - 1);
        xy1 = S.ring_xy1[slot];
        xy2 = S.ring_xy2[slot];
        u = S.ring_u[slot];
    };
    take(P.s);
    phase_end();
    for (;;) {
        // ---- terms
        const uint32_t outcome = S.ctrl[kCtrlRound];
        int32_t x1, y1, x2, y2, p1, p2, m1, m2;
        uint32_t v1, v2;
        float uniform;
        auto load = [&]() __attribute__((always_inline)) {
            x1 = (int32_t)(xy1 & 0xffffu);
            y1 = (int32_t)(xy1 >> 16);
            x2 = (int32_t)(xy2 & 0xffffu);
            y2 = (int32_t)(xy2 >> 16);
            uniform = u;
            p1 = y1 * gw + x1;
            p2 = y2 * gw + x2;
            m1 = gget(grid, p1);
            m2 = gget(grid, p2);
            v1 = S.stamp[S.at(p1)];
            v2 = S.stamp[S.at(p2)];
        };
        load();
        R.next(outcome);
        if (traced && lane < first) {  // (the last round's)
            if (job.trace_delta) gstore(job.trace_delta, it, skip ? __int_as_float(0x7fc00000) : delta);
            if (job.trace_accept) gstore(job.trace_accept, it, (uint8_t)(acc ? 1 : 0));
        }
        if (R.s >= max_iter) break;
        R.begin(S, words, kJudgeWave * 64 + lane, Nothing{}, [&]() __attribute__((always_inline)) {
            take(R.s);
            load();
        });
        it = R.s + lane;
        const uint32_t mine = (R.tag << 7) | ((uint32_t)(63 - lane) << 1);
        skip = it >= max_iter || p1 == p2 || m1 == kEmpty || m2 == kEmpty;
        const uint64_t nonskip = wave_ballot(!skip);
        float temp = 1.0f;
        if (!skip && !job.greedy) temp = gload(job.temps, kbase + lanes_before(nonskip));
        const int64_t remain = max_iter - R.s;
        first = remain < 64 ? (int32_t)remain : 64;
        if (R.hopeful) {
            first = expected_prefix(v1, v2, mine, skip, remain);
            if (!skip && lane < first) {  // (all of these cells are different)
                gput(grid, p1, m2);
                gput(grid, p2, m1);
            }
            take(R.s + first);
            if constexpr (kHbm) __threadfence();
        }
        const bool adjacent =
            p1 - p2 == gw || p2 - p1 == gw || (y1 == y2 && (x1 - x2 == 1 || x2 - x1 == 1));
        phase_end();
        // ---- decisions
        delta = m1 == m2 ? 0.0f : added_terms(S, lane, adjacent);
        acc = !skip && accepts(job, delta, temp, uniform);
        const uint64_t acc_all = wave_ballot(acc);
        const uint64_t below = first >= 64 ? ~0ull : (1ull << first) - 1ull;
        const uint64_t rejected = nonskip & ~acc_all & below;
        uint64_t commit = below;
        const bool as_expected = R.hopeful && !rejected;
        if (!as_expected) {
            bool conflict = false;
            if (R.hopeful) {
                // took a value that a rejected lane would have moved
#pragma unroll
                for (int i = 0; i < kSlotWaves; ++i) {
                    const uint32_t k = S.from[64 * i + lane];
                    conflict |= k != kNoLane && ((rejected >> (k & 63u)) & 1ull) != 0ull;
                }
            } else {
                if (acc) {
                    atomicMax(&S.stamp[S.at(p1)], mine);
                    atomicMax(&S.stamp[S.at(p2)], mine);
                }
                // (one wave's LDS operations are done in order)
                asm volatile("" ::: "memory");
                const int32_t q[10] = {p1, p2,
                                       y1 > 0 ? p1 - gw : p1, y1 < gh - 1 ? p1 + gw : p1,
                                       x1 > 0 ? p1 - 1 : p1,  x1 < gw - 1 ? p1 + 1 : p1,
                                       y2 > 0 ? p2 - gw : p2, y2 < gh - 1 ? p2 + gw : p2,
                                       x2 > 0 ? p2 - 1 : p2,  x2 < gw - 1 ? p2 + 1 : p2};
#pragma unroll
                for (int i = 0; i < 10; ++i) conflict |= S.stamp[S.at(q[i])] > (mine | 1u);
            }
            const uint64_t c = wave_ballot(conflict && !skip);
            const int32_t expected = first;
            first = min(first, c ? __ffsll((unsigned long long)c) - 1 : 64);
            commit = first >= 64 ? ~0ull : (1ull << first) - 1ull;
            const bool keep = lane_in(acc_all & commit);
            if (R.hopeful ? !skip && lane < expected && !keep : keep) {
                // (hopeful: back; else no lower lane of this round wrote p1 or p2)
                gput(grid, p1, R.hopeful ? m1 : m2);
                gput(grid, p2, R.hopeful ? m2 : m1);
            }
            if constexpr (kHbm) __threadfence();
        }
        const uint64_t accmask = acc_all & commit;
        // the accepted deltas for the cost wave (adding +0.0 changes no sum)
        S.pack[lane] = lane_in(accmask) ? delta : 0.0f;
        const int32_t n_acc = __popcll(accmask), n_ev = __popcll(nonskip & commit);
        lean = (lean - (lean >> 3)) + (9 * n_acc - 5 * n_ev);
        if (lane == 0)
            S.ctrl[kCtrlRound] =
                pack_round(first, !job.greedy && lean >= 0, !as_expected, n_acc);
        accepted += n_acc;
        evaluated += n_ev;
        kbase += n_ev;
        ++rounds;
        if (R.hopeful) ++R.tag;  // (the slot waves' reads)
        phase_end();
    }
    out->accepted = accepted;
    out->evaluated = evaluated;
    out->rounds = rounds;
}

// The draw waves, in the decisions phase, whose slot waves leave their SIMDs
// the most: the 64 proposals behind the `filled` first.  filled >= s + 128
// holds in every round before its terms (they look at proposals up to there),
// and a block only overwrites slots before s (filled <= s + 192).
template <typename G>
__device__ __forceinline__ void draw_wave(const AnnealJob& job, const AnnealShared<G>& S, int w,
                                          int lane, int32_t words, const Progress& P) {
    Rounds R;
    R.s = P.s;
    R.hopeful = !job.greedy;
    const uint32_t k = w == kDraw1Wave ? 0u : 2u;
    uint32_t* const ring = w == kDraw1Wave ? S.ring_xy1 : S.ring_xy2;
    int64_t filled = P.s + kRing;
    phase_end();
    for (;;) {
        R.next(S.ctrl[kCtrlRound]);
        if (R.s >= job.max_iter) return;
        R.begin(S, words, w * 64 + lane, Nothing{}, Nothing{});
        phase_end();
        if (filled <= R.s + kRing - 64) {
            const uint64_t j = (uint64_t)(filled + lane);
            ring[j & (kRing - 1)] = (uint32_t)draw_range(job.seed, j, k, job.grid_w) |
                                    (uint32_t)draw_range(job.seed, j, k + 1, job.grid_h) << 16;
            filled += 64;
        }
        if (R.hopeful) ++R.tag;
        phase_end();
    }
}

// The running cost: a round's deltas in proposal order, +0.0 for those not
// accepted.
struct CostSum {
    float cost, best;
    int64_t improved;
    float c;  // each lane's sum in the round being added
    template <typename G>
    __device__ __forceinline__ void load(const AnnealShared<G>& S) {
        cost = __uint_as_float(uniform_copy(S.ctrl[kCtrlCost]));
        best = __uint_as_float(uniform_copy(S.ctrl[kCtrlBest]));
        improved = uniform_copy(reinterpret_cast<const int64_t*>(S.ctrl)[kCtrlImproved / 2]);
    }
    template <typename G>
    __device__ __forceinline__ void store(const AnnealShared<G>& S) const {
        S.ctrl[kCtrlCost] = __float_as_uint(cost);
        S.ctrl[kCtrlBest] = __float_as_uint(best);
        reinterpret_cast<int64_t*>(S.ctrl)[kCtrlImproved / 2] = improved;
    }
    __device__ __forceinline__ void add(const float* pack, int lane) {
        c = add_lanes(cost, pack[lane], lane);
    }
    __device__ __forceinline__ void count(int32_t n_acc, bool greedy) {
        if (greedy) {  // optimize_greedy counts every accepted swap
            improved += n_acc;
        } else if (wave_ballot(c < best)) {
            // new bests: below the best before the round and all sums before
            const float p = wave_scan_min(__builtin_fminf(c, best));
            const float before = __int_as_float(__builtin_amdgcn_update_dpp(
                __float_as_int(best), __float_as_int(p), 0x138, 0xF, 0xF, false));  // the lane below's
            improved += __popcll(wave_ballot(c < before));
            best = readlane_f(p, 63);
        }
    }
};

// The cost wave; it also draws u for the draw waves' blocks.
template <typename G>
__device__ __forceinline__ void cost_wave(const AnnealJob& job, const AnnealShared<G>& S, int lane,
                                          int32_t words, const Progress& P) {
    Rounds R;
    R.s = P.s;
    R.hopeful = !job.greedy;
    CostSum C;
    C.load(S);
    int64_t filled = P.s + kRing;
    phase_end();
    for (;;) {
        R.next(S.ctrl[kCtrlRound]);
        if (R.s >= job.max_iter) break;
        R.begin(S, words, kCostWave * 64 + lane, Nothing{}, Nothing{});
        if (R.pending) C.add(S.pack, lane);
        phase_end();
        if (R.pending) C.count(R.pending, job.greedy != 0);
        if (filled <= R.s + kRing - 64) {
            const uint64_t j = (uint64_t)(filled + lane);
            S.ring_u[j & (kRing - 1)] = draw_unit(job.seed, j);
            filled += 64;
        }
        if (R.hopeful) ++R.tag;
        phase_end();
    }
    if (R.pending) {
        C.add(S.pack, lane);
        C.count(R.pending, job.greedy != 0);
    }
    if (lane == 0) C.store(S);
}

// ----------------------------------------------------------- whole blocks
// While nearly all proposals are accepted (annealing starts hot), a block of
// 64 need not end at the first swap that meets an earlier one's cell: if all
// of them are taken to be accepted, what a lane's cells hold before its swap
// follows from the swaps below it.  Every lane sets its bit in both its
// cells' words.  The highest bit below a lane's own in a cell's word is the lane
// k that wrote it last, and what k wrote is what k's other cell held before: a
// pointer to one of 128 nodes (a lane, and 64 for its second cell).  The
// pointers lead to ever lower lanes and end at a node whose cell nobody wrote,
// so doubling them finds every node's origin, the cell of the grid that holds
// its material, in log2 of the longest chain steps (two or three).  A block
// commits the lanes before its first rejected one, and that one.
//
// Two phases a block: in the first the slot waves read the grid at the origins
// and make terms, while a marking wave sets the bits of the next block; in the
// second the judge decides and commits, while the marking wave finds the next
// block's origins (which no commit changes).  After a rejection the judge sets
// the bits anew, and a third phase finds the origins.
//
// A block takes 1.8 us: 1,600 cycles of terms, 2,100 of decisions (the judge
// alone: sums, test, commit), 400 of reading the outcome.  With every slot wave
// finding all origins for itself 1.9; with one table, set and read in the decisions,
// 1.8 and no better at 300 cells, but 2.0 at 4,800; with tables that cells share,
// for grids of any size, 2.1 (20,000 proposals on 200 x 120 cells 782 us).
struct Touch {
    uint64_t* words;  // [2][cells]
    int32_t cells;
    __device__ __forceinline__ uint64_t* of(int32_t block, int32_t p) const {
        return &words[(block & 1) * cells + p];
    }
};
// (every lane takes part: it has another lane's value)
__device__ __forceinline__ int32_t from_lane(int32_t v, uint32_t k) {
    return __builtin_amdgcn_ds_bpermute((int32_t)(k << 2), v);
}
// The origins of a block's nodes, and its materials, in `from`'s place.
constexpr int32_t kOrigins = 128;

// A block's proposals: what they are, and their bits.
struct Proposals {
    uint32_t xy1, xy2;
    float u;
    int32_t p1, p2;
    bool skip;
    template <typename G>
    __device__ __forceinline__ void take(const AnnealJob& job, const AnnealShared<G>& S, G* grid,
                                         int64_t it) {
        const uint32_t slot = (uint32_t)it & (kRing - 1);
        xy1 = S.ring_xy1[slot];
        xy2 = S.ring_xy2[slot];
        u = S.ring_u[slot];
        p1 = (int32_t)(xy1 >> 16) * job.grid_w + (int32_t)(xy1 & 0xffffu);
        p2 = (int32_t)(xy2 >> 16) * job.grid_w + (int32_t)(xy2 & 0xffffu);
        // (which cells are empty never changes)
        const int32_t m1 = gget(grid, p1), m2 = gget(grid, p2);
        skip = (it >= job.max_iter) | (p1 == p2) | (m1 == kEmpty) | (m2 == kEmpty);
    }
    __device__ __forceinline__ void mark(const Touch& T, int32_t block, int lane) const {
        if (!skip) {
            atomicOr((unsigned long long*)T.of(block, p1), 1ull << lane);
            atomicOr((unsigned long long*)T.of(block, p2), 1ull << lane);
        }
    }
    __device__ __forceinline__ void clear(const Touch& T, int32_t block) const {
        if (!skip) {
            *T.of(block, p1) = 0ull;
            *T.of(block, p2) = 0ull;
        }
    }
    // Finds where the materials of all 128 nodes are.
    template <typename G>
    __device__ __forceinline__ void origins(const AnnealShared<G>& S, const Touch& T, int32_t block,
                                            int lane) const {
        const uint64_t below = (1ull << lane) - 1ull;
        const uint64_t t1 = *T.of(block, p1) & below, t2 = *T.of(block, p2) & below;
        int32_t c1 = p1, c2 = p2;
        if (wave_ballot((t1 | t2) != 0)) {
            // who wrote the cells last (nobody: this lane, for the reads), and
            // whether as its first: then it left there what its second held
            const uint32_t k1 = t1 ? 63u - (uint32_t)__builtin_clzll(t1) : (uint32_t)lane;
            const uint32_t k2 = t2 ? 63u - (uint32_t)__builtin_clzll(t2) : (uint32_t)lane;
            const int32_t f1 = from_lane(p1, k1), f2 = from_lane(p1, k2);
            uint32_t n1 = t1 ? k1 | (f1 == p1 ? 64u : 0u) : (uint32_t)lane;
            uint32_t n2 = t2 ? k2 | (f2 == p2 ? 64u : 0u) : (uint32_t)lane | 64u;
            for (uint32_t both = n1 | n2 << 8;;) {
                const uint32_t a1 = (uint32_t)from_lane((int32_t)both, n1 & 63u);
                const uint32_t a2 = (uint32_t)from_lane((int32_t)both, n2 & 63u);
                n1 = (n1 & 64u ? a1 >> 8 : a1) & 127u;
                n2 = (n2 & 64u ? a2 >> 8 : a2) & 127u;
                const uint32_t next = n1 | n2 << 8;
                if (!wave_ballot(next != both)) break;
                both = next;
            }
            const int32_t x1 = from_lane(p1, n1 & 63u), y1 = from_lane(p2, n1 & 63u);
            const int32_t x2 = from_lane(p1, n2 & 63u), y2 = from_lane(p2, n2 & 63u);
            c1 = n1 & 64u ? y1 : x1;
            c2 = n2 & 64u ? y2 : x2;
        }
        S.from[kOrigins + lane] = (uint32_t)c1;
        S.from[kOrigins + 64 + lane] = (uint32_t)c2;
    }
};

// The node that a slot wave's neighbour comes from, -1: its own cell.
__device__ __forceinline__ int32_t neighbour_node(const Touch& T, int32_t block, const Place& p,
                                                  int lane) {
    const uint64_t t = *T.of(block, p.q) & ((1ull << lane) - 1ull);
    const uint32_t k = t ? 63u - (uint32_t)__builtin_clzll(t) : (uint32_t)lane;
    const int32_t first = from_lane(p.p1, k);
    return t ? (int32_t)(k | (first == p.q ? 64u : 0u)) : -1;
}

// The rounds take over for good when the blocks, over the last sixteen or so,
// commit less than rounds do in a block's time: a round commits some 0.55
// sqrt(cells) if all is accepted, and a block takes 1.6 to 1.8 times as long.
// The mean begins a quarter above that line: a run that begins cold leaves after
// some four blocks, not after the 23 (300 cells) or 38 (48) that a mean that begins
// at 64 takes to fall (1,000 proposals on 300 cells, 8% accepted, 195 -> 152 us).
template <typename G>
__device__ __forceinline__ void follow_blocks(const AnnealJob& job, const AnnealShared<G>& S, G* grid,
                                              const Touch& T, int w, int lane, Progress& P) {
    const int32_t gw = job.grid_w;
    const int64_t max_iter = job.max_iter;
    const int32_t least =
        (int32_t)(16.0f * 0.88f * __builtin_sqrtf((float)(job.grid_w * job.grid_h)));
    int64_t filled = kRing;
    int32_t block = 0, pending = 0, added_last = 0, mean = least + least / 4;
    const bool traced = job.trace_delta || job.trace_accept;
    bool again = true;
    CostSum C;
    Place p;
    int32_t node;
    Proposals now, next;
    if (w == kJudgeWave) {
        now.take(job, S, grid, lane);
        now.mark(T, 0, lane);
    }
    if (w == kCostWave) C.load(S);
    phase_end();
    for (;;) {
        // ---- terms
        if (again) {
            if (w < kSlotWaves) {
                p = place_of(job, S, w, P.s + lane);
                node = neighbour_node(T, block, p, lane);
            } else if (w == kMarkWave) {
                next.take(job, S, grid, P.s + lane);
                next.origins(S, T, block, lane);
            }
            phase_end();
        }
        uint64_t t1, t2, nonskip;
        float temp;
        if (w < kSlotWaves) {
            const int32_t o1 = (int32_t)S.from[kOrigins + lane],
                          o2 = (int32_t)S.from[kOrigins + 64 + lane],
                          on = (int32_t)S.from[kOrigins + max(node, 0)];
            const int32_t oa = node < 0 ? p.q : on;
            const int32_t m1 = gget(grid, o1), m2 = gget(grid, o2), a = gget(grid, oa);
            if (w == 0) {
                S.from[lane] = (uint32_t)m1;
                S.from[64 + lane] = (uint32_t)m2;
            }
            float4 l1 = make_float4(0, 0, 0, 0), l2 = l1, la = l1;
            if (S.labs) {
                if (job.n > 0) {
                    l1 = S.labs[max(m1, 0)];
                    l2 = S.labs[max(m2, 0)];
                    la = S.labs[max(a, 0)];
                }
            } else {
                // (a gather from memory takes the address unit 64 cycles: each
                // Lab once)
                if (job.n > 0) {
                    la = gload4(job.lab4, max(a, 0));
                    if ((w & 3) == 0) S.lab_m[w * 16 + lane] = gload4(job.lab4, max(w == 0 ? m1 : m2, 0));
                }
                phase_end();
                l1 = S.lab_m[lane];
                l2 = S.lab_m[64 + lane];
            }
            const bool ok = p.in && !p.self && a != kEmpty;
            const float c1 = adj_term(l1, la), c2 = adj_term(l2, la);
            reinterpret_cast<float2*>(S.terms)[((w >> 1) * 64 + lane) * 2 + (w & 1)] =
                make_float2(ok ? c1 : 0.0f, ok ? c2 : 0.0f);
            // the partner as a neighbour of the first cell: the mutual term
            if (w < 4 && p.self) S.mutual[lane] = c1;
        } else {
            if (w == kJudgeWave) {
                nonskip = wave_ballot(!now.skip);
                temp = 1.0f;
                if (!now.skip) temp = gload(job.temps, P.evaluated + lanes_before(nonskip));
                // the lanes above this one that write its cells
                const uint64_t above = ~((2ull << lane) - 1ull);
                t1 = *T.of(block, now.p1) & above;
                t2 = *T.of(block, now.p2) & above;
                next.take(job, S, grid, P.s + 64 + lane);
            } else if (w == kMarkWave) {
                next.take(job, S, grid, P.s + 64 + lane);
                next.mark(T, block + 1, lane);
            } else if (w == kCostWave && added_last) {
                C.count(added_last, false);
                added_last = 0;
            }
            if (!S.labs) phase_end();
        }
        phase_end();
        // ---- decisions
        if (w < kSlotWaves) {
            p = place_of(job, S, w, P.s + 64 + lane);
            node = neighbour_node(T, block + 1, p, lane);
        } else if (w == kMarkWave) {
            next.origins(S, T, block + 1, lane);
        } else if (w == kJudgeWave) {
            const int32_t m1 = (int32_t)S.from[lane], m2 = (int32_t)S.from[64 + lane];
            const bool adjacent =
                now.p1 - now.p2 == gw || now.p2 - now.p1 == gw ||
                ((now.xy1 >> 16) == (now.xy2 >> 16) &&
                 (now.p1 - now.p2 == 1 || now.p2 - now.p1 == 1));
            const float added = added_terms(S, lane, adjacent);
            const float delta = m1 == m2 ? 0.0f : added;
            const bool acc = !now.skip && accepts(job, delta, temp, now.u);
            const uint64_t rejected = nonskip & ~wave_ballot(acc);
            const int32_t r = rejected ? __ffsll((unsigned long long)rejected) - 1 : 64;
            const int64_t remain = max_iter - P.s;
            const int32_t end = remain < 64 ? (int32_t)remain : 64, advance = min(r + 1, end);
            const uint64_t commit = r >= 64 ? ~0ull : (1ull << r) - 1ull;
            const uint64_t done = advance >= 64 ? ~0ull : (1ull << advance) - 1ull;
            // of the committed lanes that write a cell, the last
            const bool keep = lane_in(nonskip & commit);
            if (keep && !(t1 & commit)) gput(grid, now.p1, m2);
            if (keep && !(t2 & commit)) gput(grid, now.p2, m1);
            now.clear(T, block);
            S.pack[64 * (block & 1) + lane] = keep ? delta : 0.0f;
            if (traced && lane < advance) {
                const int64_t it = P.s + lane;
                if (job.trace_delta)
                    gstore(job.trace_delta, it, now.skip ? __int_as_float(0x7fc00000) : delta);
                if (job.trace_accept) gstore(job.trace_accept, it, (uint8_t)(acc ? 1 : 0));
            }
            mean += advance - mean / 16;
            const bool stop = P.s + advance >= max_iter || mean < least;
            if (lane == 0)
                S.ctrl[kCtrlRound] = (uint32_t)advance | (stop ? 128u : 0u) |
                                     (uint32_t)__popcll(nonskip & commit) << 8 |
                                     (uint32_t)__popcll(nonskip & done) << 16;
            if (advance != 64 && !stop) {
                // (one wave's LDS operations are done in order)
                next.clear(T, block + 1);
                asm volatile("" ::: "memory");
                next.take(job, S, grid, P.s + advance + lane);
                next.mark(T, block + 1, lane);
            }
            now = next;
        } else {
            if (w == kCostWave && pending) {
                C.add(S.pack + 64 * ((block - 1) & 1), lane);
                added_last = pending;
            }
            if (filled <= P.s + kRing - 64) {
                const uint64_t j = (uint64_t)(filled + lane);
                const uint32_t slot = (uint32_t)j & (kRing - 1);
                if (w == kCostWave) {
                    S.ring_u[slot] = draw_unit(job.seed, j);
                } else {
                    S.ring_xy1[slot] = (uint32_t)draw_range(job.seed, j, 0, job.grid_w) |
                                       (uint32_t)draw_range(job.seed, j, 1, job.grid_h) << 16;
                    S.ring_xy2[slot] = (uint32_t)draw_range(job.seed, j, 2, job.grid_w) |
                                       (uint32_t)draw_range(job.seed, j, 3, job.grid_h) << 16;
                }
                filled += 64;
            }
        }
        phase_end();
        const uint32_t v = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)S.ctrl[kCtrlRound]);
        const int32_t advance = (int32_t)(v & 127u);
        P.s += advance;
        pending = (int32_t)(v >> 8 & 127u);
        P.accepted += pending;
        P.evaluated += (int64_t)(v >> 16);
        ++P.rounds;
        ++block;
        again = advance != 64;
        if (v & 128u) break;
    }
    if (w == kCostWave) {
        if (added_last) C.count(added_last, false);
        if (pending) {
            C.add(S.pack + 64 * ((block - 1) & 1), lane);
            C.count(pending, false);
        }
        if (lane == 0) C.store(S);
    }
}

// kHbm: the grid stays in HBM (the job's own grid, swapped in place), for
// grids too large for LDS.
template <typename G, bool kHbm>
__global__ __launch_bounds__(kAnnealThreads) void anneal_kernel(AnnealJob single,
                                                                const AnnealJob* __restrict__ jobs) {
    extern __shared__ __align__(16) uint32_t sm[];
    const AnnealJob job = uniform_copy(jobs ? jobs[blockIdx.x] : single);
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int32_t cells = job.grid_w * job.grid_h;
    const int32_t words = stamp_words(cells, job.blocks != 0);
    typedef typename std::conditional<kHbm, HbmGrid, G>::type Grid;
    AnnealShared<Grid> S;
    S.stamp = sm;
    S.lab_m = reinterpret_cast<float4*>(sm + words);
    S.terms = S.lab_m + 2 * 64;
    S.from = reinterpret_cast<uint32_t*>(S.terms + kSlotWaves / 2 * 64);
    S.mutual = reinterpret_cast<float*>(S.from + kFromWords);
    S.pack = S.mutual + kMutualWords;
    S.ring_xy1 = reinterpret_cast<uint32_t*>(S.pack + kPackWords);
    S.ring_xy2 = S.ring_xy1 + kRing;
    S.ring_u = reinterpret_cast<float*>(S.ring_xy2 + kRing);
    S.ctrl = S.ring_xy2 + 2 * kRing;
    S.hashed = cells > kHashStamps;
    uint32_t* const grid_at = sm + words + kFixedWords;
    const int32_t kind = kHbm ? kAnnealHbm : sizeof(G) == 2 ? kAnnealNarrow : kAnnealWide;
    float4* const labs = reinterpret_cast<float4*>(grid_at + grid_words(cells, kind));
    S.labs = job.labs_in_lds ? labs : nullptr;
    HbmGrid hbm{job.grid};
    Grid* grid;
    if constexpr (kHbm) {
        grid = &hbm;
    } else {
        grid = reinterpret_cast<G*>(grid_at);
        // (eight loads in flight)
        for (int32_t i = tid; i < cells; i += 8 * kAnnealThreads) {
            int32_t m[8];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                m[k] = gload(job.grid, min(i + k * kAnnealThreads, cells - 1));
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (i + k * kAnnealThreads < cells) grid[i + k * kAnnealThreads] = (G)m[k];
        }
    }
    if (S.labs)
        for (int32_t i = tid; i < job.n; i += 4 * kAnnealThreads) {
            float4 l[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) l[k] = gload4(job.lab4, min(i + k * kAnnealThreads, job.n - 1));
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (i + k * kAnnealThreads < job.n) labs[i + k * kAnnealThreads] = l[k];
        }
    // the next proposals (coordinates are in the grid past max_iter too)
    auto draw_ring = [&](int64_t from) {
        if (tid >= kRing) return;
        const uint64_t d = (uint64_t)(from + tid);
        const uint32_t slot = (uint32_t)d & (kRing - 1);
        S.ring_xy1[slot] = (uint32_t)draw_range(job.seed, d, 0, job.grid_w) |
                           (uint32_t)draw_range(job.seed, d, 1, job.grid_h) << 16;
        S.ring_xy2[slot] = (uint32_t)draw_range(job.seed, d, 2, job.grid_w) |
                           (uint32_t)draw_range(job.seed, d, 3, job.grid_h) << 16;
        S.ring_u[slot] = draw_unit(job.seed, d);
    };
    draw_ring(0);
    __syncthreads();
    const float initial =
        S.labs ? total_cost_block(grid, job.grid_w, job.grid_h, TermLds{S.labs}, S.stamp)
               : total_cost_block(grid, job.grid_w, job.grid_h, TermLab{job.lab4}, S.stamp);
    __syncthreads();
    for (int32_t i = tid; i < words; i += kAnnealThreads) S.stamp[i] = 0u;
    if (tid == 0) {
        S.ctrl[kCtrlCost] = S.ctrl[kCtrlBest] = __float_as_uint(initial);
        reinterpret_cast<int64_t*>(S.ctrl)[kCtrlImproved / 2] = 0;
    }
    __syncthreads();
    Progress P;
    if constexpr (!kHbm) {
        if (job.blocks && job.max_iter > 0) {
            const Touch T{reinterpret_cast<uint64_t*>(sm), cells};
            follow_blocks(job, S, grid, T, w, lane, P);
            if (P.s < job.max_iter) {
                __syncthreads();
                draw_ring(P.s);
                for (int32_t i = tid; i < words; i += kAnnealThreads) S.stamp[i] = 0u;
            }
            __syncthreads();
        }
    }
    if (tid == 0) S.ctrl[kCtrlRound] = pack_round(0, !job.greedy, false, 0);
    __syncthreads();

    AnnealOut r{};
    if (w < kSlotWaves)
        slot_wave(job, S, grid, w, lane, words, P);
    else if (w == kJudgeWave)
        judge_wave<Grid, kHbm>(job, S, grid, lane, words, P, &r);
    else if (w != kCostWave)
        draw_wave(job, S, w, lane, words, P);
    else
        cost_wave(job, S, lane, words, P);
    __syncthreads();
    if constexpr (!kHbm)
        for (int32_t i = tid; i < cells; i += kAnnealThreads) gstore(job.grid, i, (int32_t)grid[i]);
    if (tid == 64 * kJudgeWave && job.result) {
        r.initial_cost = initial;
        r.final_cost = __uint_as_float(S.ctrl[kCtrlCost]);
        r.best_cost = job.greedy ? r.final_cost : __uint_as_float(S.ctrl[kCtrlBest]);
        r.improved = reinterpret_cast<const int64_t*>(S.ctrl)[kCtrlImproved / 2];
        r.iterations = job.max_iter;
        *job.result = r;
    }
}

namespace {
size_t anneal_lds_bytes(int32_t cells, int32_t kind, int32_t labs, bool blocks) {
    return sizeof(uint32_t) *
               ((size_t)stamp_words(cells, blocks) + kFixedWords + grid_words(cells, kind)) +
           sizeof(float4) * (size_t)labs;
}
// Whole blocks commit up to 64 proposals in 1.6-1.8 us, a round some 0.55
// sqrt(cells) in 1.0.  Measured (anneal, us, rounds alone and with blocks): 300
// cells 112 and 44, 1,400 61 and 47, 4,800 84 and 81 on one picture, 79 and 82
// on another.
constexpr int32_t kFollowCells = 4096;
}  // namespace

int32_t anneal_kind(int32_t cells, int32_t n, int32_t gw, int32_t gh, size_t max_lds) {
    auto fits = [&](int32_t kind) { return anneal_lds_bytes(cells, kind, 0, false) <= max_lds; };
    if (n < 32768 && fits(kAnnealNarrow)) return kAnnealNarrow;
    if (fits(kAnnealWide)) return kAnnealWide;
    if (gw < 65536 && gh < 65536 && fits(kAnnealHbm)) return kAnnealHbm;
    return -1;
}

// The Labs have the first claim on LDS, then the blocks' tables.
AnnealLayout anneal_layout(int32_t cells, int32_t kind, int32_t n, bool greedy, bool want_labs,
                           size_t max_lds) {
    AnnealLayout l;
    l.labs = want_labs && anneal_lds_bytes(cells, kind, n, false) <= max_lds;
    l.blocks = !greedy && kind != kAnnealHbm && cells <= kFollowCells &&
               anneal_lds_bytes(cells, kind, l.labs ? n : 0, true) <= max_lds;
    l.lds = anneal_lds_bytes(cells, kind, l.labs ? n : 0, l.blocks);
    return l;
}

namespace {
template <typename... A>
void launch_anneal(int32_t kind, dim3 grid, size_t lds_bytes, hipStream_t stream, A... args) {
    const dim3 threads(kAnnealThreads);
    if (kind == kAnnealNarrow)
        hipLaunchKernelGGL((anneal_kernel<int16_t, false>), grid, threads, lds_bytes, stream,
                           args...);
    else if (kind == kAnnealWide)
        hipLaunchKernelGGL((anneal_kernel<int32_t, false>), grid, threads, lds_bytes, stream,
                           args...);
    else
        hipLaunchKernelGGL((anneal_kernel<int32_t, true>), grid, threads, lds_bytes, stream,
                           args...);
}
}  // namespace

void launch_anneal_single(const AnnealJob& job, int32_t kind, size_t lds_bytes, hipStream_t stream) {
    launch_anneal(kind, dim3(1), lds_bytes, stream, job, (const AnnealJob*)nullptr);
}

void launch_anneal_batch(const AnnealJob* d_jobs, int32_t n_jobs, int32_t kind, size_t lds_bytes,
                         hipStream_t stream) {
    if (n_jobs <= 0) return;
    AnnealJob unused{};
    launch_anneal(kind, dim3(n_jobs), lds_bytes, stream, unused, d_jobs);
}

hipError_t anneal_configure(int max_lds) {
    const void* kernels[] = {
        reinterpret_cast<const void*>(&anneal_kernel<int16_t, false>),
        reinterpret_cast<const void*>(&anneal_kernel<int32_t, false>),
        reinterpret_cast<const void*>(&anneal_kernel<int32_t, true>),
    };
    for (const void* k : kernels) {
        const hipError_t e = raise_dynamic_lds(k, max_lds);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// ------------------------------------------------ cost / delta / penalty
__global__ __launch_bounds__(kAnnealThreads) void total_cost_kernel(
    const int32_t* __restrict__ grid, int32_t gw, int32_t gh, const float4* __restrict__ lab4,
    float* __restrict__ out) {
    __shared__ __align__(16) uint32_t lds[kCostWords];
    const float t = total_cost_block(grid, gw, gh, TermLab{lab4}, lds);
    if (threadIdx.x == 0) *out = t;
}

void launch_total_cost(const int32_t* grid, int32_t gw, int32_t gh, const float4* lab4, float* out,
                       hipStream_t stream) {
    hipLaunchKernelGGL(total_cost_kernel, dim3(1), dim3(kAnnealThreads), 0, stream, grid, gw, gh,
                       lab4, out);
}

__global__ void swap_delta_kernel(const int32_t* __restrict__ grid, int32_t gw, int32_t gh,
                                  const float4* __restrict__ lab4,
                                  const int32_t* __restrict__ pairs, int32_t p,
                                  float* __restrict__ out) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= p) return;
    const int32_t* q = pairs + 4 * (int64_t)i;
    out[i] = swap_delta_dev(grid, gw, gh, lab4, q[0], q[1], q[2], q[3]);
}

void launch_swap_deltas(const int32_t* grid, int32_t gw, int32_t gh, const float4* lab4,
                        const int32_t* pairs, int32_t p, float* out, hipStream_t stream) {
    if (p <= 0) return;
    hipLaunchKernelGGL(swap_delta_kernel, dim3((p + 255) / 256), dim3(256), 0, stream, grid, gw, gh,
                       lab4, pairs, p, out);
}

// calculate_penalty (src/adjacency.rs:63-88): Up, Down, Left, Right.
__global__ void penalty_kernel(const int32_t* __restrict__ grid, int32_t gw, int32_t gh,
                               const float4* __restrict__ lab4, float weight,
                               const int32_t* __restrict__ queries, int32_t nq,
                               float* __restrict__ out) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nq) return;
    const int32_t m = queries[3 * (int64_t)i], x = queries[3 * (int64_t)i + 1],
                  y = queries[3 * (int64_t)i + 2];
    const float4 lm = lab4[m];
    float p = 0.0f;
    int32_t nb[4], cnt = 0;
    if (y > 0) nb[cnt++] = (y - 1) * gw + x;
    if (y < gh - 1) nb[cnt++] = (y + 1) * gw + x;
    if (x > 0) nb[cnt++] = y * gw + x - 1;
    if (x < gw - 1) nb[cnt++] = y * gw + x + 1;
    for (int32_t j = 0; j < cnt; ++j) {
        const int32_t o = grid[nb[j]];
        if (o != kEmpty) p += adj_term(lm, lab4[o]);
    }
    out[i] = p * weight;
}

void launch_penalties(const int32_t* grid, int32_t gw, int32_t gh, const float4* lab4, float weight,
                      const int32_t* queries, int32_t nq, float* out, hipStream_t stream) {
    if (nq <= 0) return;
    hipLaunchKernelGGL(penalty_kernel, dim3((nq + 255) / 256), dim3(256), 0, stream, grid, gw, gh,
                       lab4, weight, queries, nq, out);
}

}  // namespace mh
