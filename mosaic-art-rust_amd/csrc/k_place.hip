// k_place.hip -- greedy placement chain (generate_mosaic's cell loop,
// src/main.rs:529-545, driving find_and_use_best_tile_with_position
// :335-418 and fallback_tile_selection :420-475, with UsageTracker
// src/lib.rs:57-89, can_place_at_position :309-333 and
// AdjacencyPenaltyCalculator::calculate_penalty src/adjacency.rs:63-88).
//
// The chain is sequential across cells (global usage counts, a global usage
// reset, and the just-placed neighbours).  Per cell there are K <= 100
// candidates: usage < max, neighbour ban, weighted penalty (similarities
// recomputed from Labs -- bit-identical to the stored matrix), score =
// sqdist + penalty; the reference's first strict-< winner is the minimum of
// (score, rank).  Many jobs run as many independent workgroups.
//
// The GUI generator's variant (src/gui/app_full.rs:1396-1563) scores
// sqrt(sqdist) + penalty with everything else unchanged: its candidate rows
// hold the square roots (k_topk.hip), and nothing here differs.
//
// Three kernels:
//  * place_raster_kernel -- what generate_mosaic runs: raster order from an
//    empty grid, so only Up and Left can be filled.  One workgroup per job:
//    a chain wave, and waves that prepare its candidates (below).
//  * place_outputs_kernel -- the distances and scores of such a run's cells,
//    after it, where the caller wants them.
//  * place_chain_kernel -- any cell order over a pre-filled grid and usage
//    (find_and_use_best_tile_with_position at arbitrary cells), one wave;
//    grid and usage in LDS, all four neighbours read per cell.  Its HBM form
//    (launched with no LDS) keeps grid and counts in the job's own buffers,
//    for libraries whose counts do not fit LDS; it also runs the raster order
//    then.
#include "mh_device.hpp"
#include "mh_kernels.hpp"

namespace mh {

// ------------------------------------------------------------ general chain
// State access of the general chain: grid and usage counts in LDS, or (kHbm,
// for libraries whose counts do not fit LDS) the job's own buffers in HBM,
// read and written with agent-scope atomics so no lane sees a stale cache
// line of a word another lane has just written.
template <bool kHbm>
struct ChainState {
    int32_t* grid;
    uint32_t* usage;
    __device__ __forceinline__ int32_t cell(int32_t i) const {
        if constexpr (kHbm)
            return __hip_atomic_load((MH_GAS int32_t*)grid + i, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
        else
            return grid[i];
    }
    __device__ __forceinline__ void set_cell(int32_t i, int32_t v) const {
        if constexpr (kHbm)
            __hip_atomic_store((MH_GAS int32_t*)grid + i, v, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        else
            grid[i] = v;
    }
    __device__ __forceinline__ uint32_t count(int32_t m) const {
        if constexpr (kHbm)
            return __hip_atomic_load((MH_GAS uint32_t*)usage + m, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
        else
            return usage[m];
    }
    __device__ __forceinline__ void set_count(int32_t m, uint32_t v) const {
        if constexpr (kHbm)
            __hip_atomic_store((MH_GAS uint32_t*)usage + m, v, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        else
            usage[m] = v;
    }
    // every lane's writes before every lane's later reads
    __device__ __forceinline__ void sync() const {
        if constexpr (kHbm) __threadfence();
        __syncthreads();
    }
};

template <bool kHbm>
__global__ __launch_bounds__(64) void place_chain_kernel(PlaceJob single,
                                                         const PlaceJob* __restrict__ jobs) {
    extern __shared__ int32_t sm[];
    const PlaceJob job = uniform_copy(jobs ? jobs[blockIdx.x] : single);
    const int lane = threadIdx.x;
    const int32_t gw = job.grid_w, gh = job.grid_h, n = job.n;
    const int32_t cells = gw * gh;
    ChainState<kHbm> S;
    if constexpr (kHbm) {
        S.grid = job.grid;
        S.usage = job.usage;
        if (job.zero_usage)
            for (int32_t i = lane; i < n; i += 64) S.set_count(i, 0u);
    } else {
        S.grid = sm;
        S.usage = reinterpret_cast<uint32_t*>(sm + cells);
        for (int32_t i = lane; i < cells; i += 64) S.grid[i] = gload(job.grid, i);
        for (int32_t i = lane; i < n; i += 64)
            S.usage[i] = job.zero_usage ? 0u : gload(job.usage, i);
    }
    S.sync();

    const int32_t K = n < kMaxCand ? n : kMaxCand;
    const uint32_t max_usage = (uint32_t)job.max_usage;
    const float weight = job.weight;
    const bool use_pen = weight > 0.0f;
    int32_t st_main = 0, st_ban = 0, st_near = 0, st_resets = 0, st_empty = 0;
    const int32_t steps = job.order ? job.n_order : cells;

    for (int32_t c = 0; c < steps; ++c) {
        const int32_t cell = job.order ? gload(job.order, c) : c;
        if (n == 0) {
            ++st_empty;
            continue;
        }
        const int32_t x = cell % gw, y = cell / gw;
        // neighbours in get_adjacent_positions order: Up, Down, Left, Right
        const int32_t nb_up = y > 0 ? S.cell(cell - gw) : kEmpty;
        const int32_t nb_down = y < gh - 1 ? S.cell(cell + gw) : kEmpty;
        const int32_t nb_left = x > 0 ? S.cell(cell - 1) : kEmpty;
        const int32_t nb_right = x < gw - 1 ? S.cell(cell + 1) : kEmpty;
        float4 lu = make_float4(0, 0, 0, 0), ld = lu, ll = lu, lr = lu;
        if (use_pen) {
            if (nb_up != kEmpty) lu = gload4(job.lab4, nb_up);
            if (nb_down != kEmpty) ld = gload4(job.lab4, nb_down);
            if (nb_left != kEmpty) ll = gload4(job.lab4, nb_left);
            if (nb_right != kEmpty) lr = gload4(job.lab4, nb_right);
        }
        const uint64_t* crow = reinterpret_cast<const uint64_t*>(job.cand) + (int64_t)cell * kCandStride;

        uint64_t best = ~0ull;
        bool placeable[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int32_t r = lane + 64 * s;
            placeable[s] = false;
            if (r < K) {
                const uint64_t rec = gload(crow, r);
                const int32_t m = (int32_t)(uint32_t)rec;
                const float dm = __uint_as_float((uint32_t)(rec >> 32));
                const bool pl = m != nb_up && m != nb_down && m != nb_left && m != nb_right;
                placeable[s] = pl;
                if (pl && S.count(m) < max_usage) {
                    float pen = 0.0f;
                    if (use_pen) {
                        const float4 lm = gload4(job.lab4, m);
                        float p = 0.0f;
                        if (nb_up != kEmpty) p += adj_term(lm, lu);
                        if (nb_down != kEmpty) p += adj_term(lm, ld);
                        if (nb_left != kEmpty) p += adj_term(lm, ll);
                        if (nb_right != kEmpty) p += adj_term(lm, lr);
                        pen = p * weight;
                    }
                    const float score = dm + pen;
                    const uint64_t key = ((uint64_t)__float_as_uint(score) << 32) | (uint32_t)r;
                    best = key < best ? key : best;
                }
            }
        }
        best = wave_min_u64(best);
        int32_t rank, stage;
        if (best != ~0ull) {
            rank = (int32_t)(best & 0xffffffffu);
            stage = 0;
            ++st_main;
        } else {
            // fallback_tile_selection: reset every usage count, then the first
            // candidate passing the neighbour ban, else nearest_one.
            for (int32_t i = lane; i < n; i += 64) S.set_count(i, 0u);
            ++st_resets;
            const uint64_t b0 = wave_ballot(placeable[0]);
            const uint64_t b1 = wave_ballot(placeable[1]);
            if (b0) {
                rank = __ffsll((unsigned long long)b0) - 1;
                stage = 1;
                ++st_ban;
            } else if (b1) {
                rank = 64 + __ffsll((unsigned long long)b1) - 1;
                stage = 1;
                ++st_ban;
            } else {
                rank = 0;
                stage = 2;
                ++st_near;
            }
        }
        const uint64_t wrec = gload(crow, rank);
        const int32_t w = (int32_t)(uint32_t)wrec;
        const float wd = __uint_as_float((uint32_t)(wrec >> 32));
        S.sync();
        if (lane == 0) {
            S.set_count(w, S.count(w) + 1u);
            S.set_cell(cell, w);
            if (job.stage) gstore(job.stage, cell, (uint8_t)stage);
            if (job.dist) gstore(job.dist, cell, wd);
            if (job.score)
                gstore(job.score, cell, stage == 0 ? __uint_as_float((uint32_t)(best >> 32)) : wd);
        }
        S.sync();
    }

    if constexpr (!kHbm) {
        for (int32_t i = lane; i < cells; i += 64) gstore(job.grid, i, S.grid[i]);
        for (int32_t i = lane; i < n; i += 64) gstore(job.usage, i, S.usage[i]);
    }
    if (lane == 0 && job.stats) {
        gstore(job.stats, 0, st_main + st_ban + st_near);
        gstore(job.stats, 1, st_main);
        gstore(job.stats, 2, st_ban);
        gstore(job.stats, 3, st_near);
        gstore(job.stats, 4, st_resets);
        gstore(job.stats, 5, st_empty);
    }
}

// ------------------------------------------------------------- raster chain
// What bounds it is the latency of one decision after another, so the chain
// wave is left with nothing but the decision: the other waves of its
// workgroup turn each candidate row, ahead of time, into a list of the
// candidates that can still win, and the chain wave picks from the lists.
//
//   * Preparing waves (prep_waves): for cells two to four groups ahead, a
//     row's candidates that are not exhausted and are not the up neighbour
//     are written to LDS, compacted in rank order (a count only grows between
//     resets, so what a stale count rules out stays out).  A list entry
//     carries a flag, "unsafe": the next entry lies within the largest
//     penalty this one can have, so it may lose although it comes first.
//   * The chain wave (chain_wave): the first entry of the list that is not
//     exhausted by now and not the left neighbour; when it is not flagged it
//     wins.  Per cell: a compare, a mask, a find-first, a lane read, a branch,
//     the commit, and the reads ahead for the next cells.
//   * One wave moves the winners from LDS to the grid.
//
// Groups of kGroup cells pass through three LDS slots; a barrier per group
// (a period) hands a slot on.  In the period in which the chain works on
// group g, the preparing waves fill group g + 2's slot, so the chain's reads
// ahead into group g + 1 never wait.  A usage reset makes the lists prepared
// before it wrong (they lack candidates that can be used again): the chain
// then ends the period and the preparation starts over from the next cell.
//
// Measured, one job at a time, against one wave that did all of it (a step of
// 450 cycles, a full evaluation in 10% of the cells): 1,500 materials in 80 x
// 60 cells 905 -> 271 us, 10,000 in 160 x 150 4,957 -> 1,867, 500 in 50 x 28
// 269 -> 89, 1,000 in 20 x 15 58 -> 30, 777 in 97 x 41 with the GUI score
// 2,283 -> 482.  A step takes 42-48 ns, and the preparation of two cells 1,350
// cycles of its wave, about a period; 0.6% (1,500 materials) to 16% (GUI
// score, whose distances lie closer) of the cells are flagged, at 0.4-1 us.
// Twelve preparing waves of a cell each: 267 us for the first, and twice the
// waves beside other jobs' work.
constexpr int32_t kGroup = 12;       // cells per period
constexpr int32_t kSlots = 3;        // groups in LDS: worked on, ready, being filled
constexpr int32_t kPrepWaves = 6;    // two cells each per period
constexpr int32_t kPrepCells = kGroup / kPrepWaves;
// Wave 0 is the chain, wave 4 stores winners (its SIMD is the chain's, so
// it gets the least work), the others prepare.
constexpr int32_t kChainThreads = 64 * (kPrepWaves + 2);
constexpr int32_t kStoreWave = 4;
// A slot: the lists' entries, those of three consecutive cells side by side
// (16 bytes a lane, the last word unused: one LDS read gives the chain three
// cells), then their distances.
constexpr int32_t kTriple = 3;
constexpr int32_t kEntryWords = kGroup / kTriple * 64 * 4;
constexpr int32_t kSlotWords = kEntryWords + kGroup * 64;
__device__ __forceinline__ int32_t entry_word(int32_t k, int32_t lane) {
    return k / kTriple * 256 + lane * 4 + k % kTriple;
}
__device__ __forceinline__ int32_t dist_word(int32_t k, int32_t lane) {
    return kEntryWords + k * 64 + lane;
}
// Materials are held as entry ids (m + 1) * 4, the byte offset of their
// count word: 0 is "none", whose word (the guard) is above every limit.
// A count word is the use count in the upper half and, in the lower, the
// material's largest adjacency term to another material as a bfloat16 rounded
// up: the preparation gets both with one LDS read, and words compare with
// limit << 16 like counts with the limit.  (Gathered from memory, the terms
// cost more than all of the preparation: a gather takes the address unit 64
// cycles.)  Counts that may not fit 16 bits are held whole, with 1 for every
// term.
constexpr uint32_t kGuard = 0xffffffffu;
__device__ __forceinline__ bool packs(const PlaceJob& job) {
    return job.zero_usage && job.max_usage < 65536;
}
// An entry's flags: kFlagged with either of kFirst (its cell is the first of
// a row) and kUnsafe.
constexpr uint32_t kFlagged = 0x80000000u, kFirst = 0x40000000u;
constexpr int32_t kUnsafeBit = 29;
constexpr uint32_t kUnsafe = 1u << kUnsafeBit;
constexpr uint32_t kEntryId = kUnsafe - 1u;
__device__ __forceinline__ uint32_t entry_id(int32_t m) { return ((uint32_t)m + 1u) * 4u; }
// f >= 0 as a bfloat16 rounded up (in the upper half of a float).
__device__ __forceinline__ uint32_t bf16_up(float f) {
    return (__float_as_uint(f) + 0xffffu) & 0xffff0000u;
}
__device__ __forceinline__ int32_t entry_material(uint32_t a) { return (int32_t)(a >> 2) - 1; }

// Winners are kept in an LDS ring until the row below has used them.  kUpPrep
// (grids at least 4 groups wide): the preparing waves read the up neighbours,
// the ring covers a row and the groups in flight.  kUpChain (3 columns to
// that): the up neighbour may be decided after the row is prepared, so the
// chain itself bans it.
constexpr int kUpPrep = 0, kUpChain = 1;
constexpr int32_t kUpPrepColumns = 4 * kGroup;
constexpr int32_t kUpRing = 128;
static_assert(kUpPrepColumns + 6 * kGroup < kUpRing,
              "kUpChain's ring covers a row and two cycles");
__host__ __device__ __forceinline__ int32_t ring_words(int32_t grid_w) {
    return grid_w >= kUpPrepColumns ? grid_w + 5 * kGroup : kUpRing;
}
// (not monotone in the width: kUpPrepColumns wide grids have the shortest)
constexpr int32_t kLeastRingColumns = kUpPrepColumns;
static_assert(kUpPrepColumns + 5 * kGroup <= kUpRing, "kLeastRingColumns");

// LDS of the chain, in words: events, guard and counts, lane scratch, winner
// ring, prepared rows, lists in preparation, material Labs (where they fit).
// The counts' place is a constant, so that it goes into the offset field of
// the chain's LDS instructions.
constexpr int32_t kEvents = 4;
constexpr int32_t kCountsAt = kEvents;
__host__ __device__ __forceinline__ int32_t scratch_at(int32_t n) {
    return kCountsAt + 1 + (n > 0 ? n : 1);
}
__host__ __device__ __forceinline__ int32_t ring_at(int32_t n) { return scratch_at(n) + 64; }
__host__ __device__ __forceinline__ int32_t rows_at(int32_t grid_w, int32_t n) {
    return (ring_at(n) + ring_words(grid_w) + 3) & ~3;
}

// Three periods, one for each slot, make a cycle; the chain leaves one event
// a cycle: 0 it worked on to the end, kDone it reached the end of the grid,
// else 1 + the cell to start over from.  (It is read at the end of the cycle
// only, so that the preparing waves' three periods are straight-line code:
// with an exit after each, the compiler waits for rows that are still in
// flight.)  After an event the chain is idle to the end of the cycle and
// through the first two periods of the next.
constexpr uint32_t kDone = 0xffffffffu;

constexpr int32_t kStageWords = 65 * 2;  // a list in preparation, see prep_cells
__host__ __device__ __forceinline__ int32_t labs_at(int32_t grid_w, int32_t n) {
    return rows_at(grid_w, n) + kSlots * kSlotWords + kGroup * kStageWords;
}

struct ChainShared {
    uint32_t* scratch; // one word per lane of the chain wave
    uint32_t* events;  // kEvents words, by cycle
    uint32_t* ring;    // entry ids of the latest winners
    uint32_t* counts;  // guard, then the n usage counts
    uint32_t* rows;    // kSlots x kSlotWords
    uint32_t* stage;   // kStageWords per list in preparation
    float4* labs;      // the material Labs, or nullptr (read from memory)
    int32_t ring_n;
};

// End of a period: this wave's LDS operations are complete (drain: the
// chain's need not be, see chain_wave), then all waves meet.
__device__ __forceinline__ void period_end(bool drain) {
    if (drain) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ uint32_t read_event(const ChainShared& S, uint32_t cycle) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)S.events[cycle & (kEvents - 1)]);
}

// i mod m for a uniform i >= -m.
__device__ __forceinline__ int32_t wrap(int32_t i, int32_t m) { return i < 0 ? i + m : i; }

// ------------------------------------------------------------ preparation
// f(Slot<0>{}), ..., f(Slot<N - 1>{}) in order, each with its index as a
// compile-time constant.
template <int I>
struct Slot {
    static constexpr int value = I;
};

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(Slot<I>{});
        static_for<I + 1, N>(f);
    }
}

// More cycles than any run has (every cycle decides at least one cell): the
// other waves' way out if they never saw the chain's last event.
__device__ __forceinline__ uint32_t cycle_cap(int32_t cells) { return (uint32_t)cells + 16u; }

struct RawRow {
    uint64_t r0, r1;  // records of ranks lane, lane + 64
};

__device__ __forceinline__ RawRow load_row(const PlaceJob& job, int32_t cell, int32_t cells, int lane) {
    const int32_t row = cell < cells ? cell : cells - 1;
    const uint64_t* rec = reinterpret_cast<const uint64_t*>(job.cand) + (int64_t)row * kCandStride;
    return RawRow{gload(rec, lane), gload(rec, lane + 64)};
}

// The rows of cells c .. c + kPrepCells - 1, from one address (at the grid's end
// those of its last cells: a cell inside reads its own).
__device__ __forceinline__ void load_rows(const PlaceJob& job, int32_t c, int32_t cells, int lane,
                                          RawRow (&q)[kPrepCells]) {
    if (c + kPrepCells <= cells) {
        const uint64_t* rec = reinterpret_cast<const uint64_t*>(job.cand) + (int64_t)c * kCandStride;
#pragma unroll
        for (int k = 0; k < kPrepCells; ++k)
            q[k] = RawRow{gload(rec, k * kCandStride + lane), gload(rec, k * kCandStride + lane + 64)};
    } else {
#pragma unroll
        for (int k = 0; k < kPrepCells; ++k) q[k] = load_row(job, c + k, cells, lane);
    }
}

// Whether the lists leave out exhausted candidates.  Those of a library of at
// most 64 materials hold every candidate without that, and stay valid across
// resets (one every n * limit cells at the least); with a limit of 0 every
// cell resets.  In all other cases a reset is at least 65 cells from the
// last one (but for counts that a caller has set).
__device__ __forceinline__ bool filters(const PlaceJob& job) {
    return (job.n > 64 && job.max_usage > 0) || !job.zero_usage;
}

// Row-constant inputs of the preparation.
struct PrepArgs {
    uint32_t limit;       // candidates whose count word is below it are kept
    bool packed;          // count words hold terms
    float w2;             // 2 * weight (doubling is exact: t * w2 is 2 t * w);
                          // -inf without a penalty: no entry has any reach
};

// A cell's list has at least this many entries, if its row has them: ranks 64
// and up are only looked at when fewer of the first 64 are kept (of one of
// the cells prepared together).  The list's last entry is reached only where
// the cells since (36 at most) took all before it; the cell then reads its
// row.  With all ranks in every list 316 us instead of 279 (1,500 materials,
// 80 x 60 cells).
constexpr uint32_t kEnough = 8;

// The kept candidates' places in a list in preparation, lanes of `kept` in
// order from `first`; a 65th place for the others.  (Branch-free: left to
// itself the compiler puts the counting under an exec mask.)
__device__ __forceinline__ uint32_t list_place(uint64_t kept, uint32_t first) {
    uint32_t p = first + lanes_before(kept);
    asm("" : "+v"(p));
    return lane_in(kept) ? p : 64u;
}

// The lists of cells c .. c + kPrepCells - 1, side by side so that their LDS
// reads are in flight together: a cell's count-limited candidates without the
// up neighbour up[k] (an entry id, 0: none), the first 64 of them.  An
// entry's reach is the largest score it can have: each of its two terms is at
// most its material's largest term to another material, t (its neighbours
// are other materials, or it would be banned), so its penalty is at most
// fl(2 t w) and its score at most fl(d + fl(2 t w)); a later entry's score is
// at least its distance.  stage: the candidates kept, by place in the list,
// {material + 1 | term << 16, distance} (the counts fit LDS, so a material
// fits 16 bits).  The distances behind a list's end bound those of the row's
// other candidates from below.  Cells past the grid get an empty list.
__device__ __forceinline__ void prep_cells(const RawRow (&q)[kPrepCells], int32_t c, int32_t cells,
                                           const uint32_t (&up)[kPrepCells],
                                           const bool (&first)[kPrepCells], const PrepArgs& P,
                                           const ChainShared& S, uint32_t* slot, int32_t k0,
                                           uint32_t* stage, int lane) {
    uint32_t m0[kPrepCells], u0[kPrepCells];
#pragma unroll
    for (int k = 0; k < kPrepCells; ++k) {
        m0[k] = (uint32_t)q[k].r0 + 1u;
        u0[k] = S.counts[m0[k]];
    }
    uint64_t b0[kPrepCells];
    uint32_t total[kPrepCells];
    bool whole = false;  // the lists hold their rows' every kept candidate, or 64
#pragma unroll
    for (int k = 0; k < kPrepCells; ++k) {
        // (ranks past the row's end read the guard)
        b0[k] = lanes_ult(u0[k], P.limit) & lanes_ne((int32_t)m0[k], (int32_t)(up[k] >> 2));
        total[k] = (uint32_t)__popcll(b0[k]);
        whole = whole || total[k] < kEnough;
    }
#pragma unroll
    for (int k = 0; k < kPrepCells; ++k) {
        uint64_t* at = reinterpret_cast<uint64_t*>(stage + k * kStageWords);
        at[list_place(b0[k], 0u)] =
            (q[k].r0 & 0xffffffff00000000ull) | ((P.packed ? u0[k] : 0x3f80u) << 16 | m0[k]);
    }
    float tail[kPrepCells];  // behind the list: rank 64, or nothing
#pragma unroll
    for (int k = 0; k < kPrepCells; ++k)
        tail[k] = readlane_f(__uint_as_float((uint32_t)(q[k].r1 >> 32)), 0);
    uint64_t end = 0ull;  // the lanes whose list may end there
    if (whole) {
        end = ~0ull;
        uint32_t m1[kPrepCells], u1[kPrepCells];
#pragma unroll
        for (int k = 0; k < kPrepCells; ++k) {
            m1[k] = (uint32_t)q[k].r1 + 1u;
            u1[k] = S.counts[m1[k]];
        }
#pragma unroll
        for (int k = 0; k < kPrepCells; ++k) {
            const uint64_t b1 =
                lanes_ult(u1[k], P.limit) & lanes_ne((int32_t)m1[k], (int32_t)(up[k] >> 2));
            uint64_t* at = reinterpret_cast<uint64_t*>(stage + k * kStageWords);
            at[min(list_place(b1, total[k]), 64u)] =
                (q[k].r1 & 0xffffffff00000000ull) | ((P.packed ? u1[k] : 0x3f80u) << 16 | m1[k]);
            total[k] += (uint32_t)__popcll(b1);
            tail[k] = __builtin_inff();
        }
    }
    if (c + kPrepCells > cells)
#pragma unroll
        for (int k = 0; k < kPrepCells; ++k) total[k] = c + k < cells ? total[k] : 0u;
    asm volatile("" ::: "memory");  // (a wave's LDS operations are done in order)
    uint64_t e[kPrepCells], en[kPrepCells];
#pragma unroll
    for (int k = 0; k < kPrepCells; ++k) {
        const uint64_t* at = reinterpret_cast<const uint64_t*>(stage + k * kStageWords) + lane;
        e[k] = at[0];
        en[k] = at[1];
    }
    // flag the entries that a later one could beat; the last place stands
    // for everything beyond it
#pragma unroll
    for (int k = 0; k < kPrepCells; ++k) {
        const uint32_t x = (uint32_t)e[k];
        const uint64_t in = lanes_ult((uint32_t)lane, total[k]);
        const float d = __uint_as_float((uint32_t)(e[k] >> 32));
        const float dn = __uint_as_float((uint32_t)(en[k] >> 32));
        const float reach = d + __uint_as_float(x & 0xffff0000u) * P.w2;
        // safe: the next beyond reach, or none next
        uint64_t safe = in >> 1 & __builtin_amdgcn_fcmpf(dn, reach, 2);  // >
        safe |= in & ~(in >> 1) & end;
        safe &= 0x7fffffffffffffffull;
        const uint32_t flags = first[k] ? kFlagged | kFirst : 0u;
        const uint32_t a = lane_in(in) ? (x & 0xffffu) << 2 : 0u;
        slot[entry_word(k0 + k, lane)] = a | flags | (lane_in(safe) ? 0u : kFlagged | kUnsafe);
        slot[dist_word(k0 + k, lane)] = __float_as_uint(lane_in(in) ? d : tail[k]);
    }
}

template <int kUp>
__device__ __forceinline__ void prep_waves(const PlaceJob& job, const ChainShared& S, int32_t v,
                                           int lane) {
    const int32_t gw = job.grid_w, cells = gw * job.grid_h;
    PrepArgs P;
    P.packed = packs(job);
    P.limit = filters(job) ? (uint32_t)job.max_usage << (P.packed ? 16 : 0) : kGuard;
    P.w2 = job.weight > 0.0f ? 2.0f * job.weight : -__builtin_inff();
    uint32_t* const stage = S.stage + v * kPrepCells * kStageWords;
    const uint32_t cap = cycle_cap(cells);
    uint32_t cycle = 0;
    int32_t start = 0;
    for (;;) {
        // rows three groups ahead are in flight in registers
        RawRow q[kSlots][kPrepCells];
        int32_t c = start + v * kPrepCells;  // this wave's first cell of the group
#pragma unroll
        for (int s = 0; s < kSlots; ++s) load_rows(job, c + s * kGroup, cells, lane, q[s]);
        // Everything landed (vmcnt 0): with nothing pending on the way in, the
        // compiler's wait counts inside the loop are those of its own loads,
        // and the rows in flight are not waited for.
        __builtin_amdgcn_s_waitcnt(0x0f70);
        int32_t x = c % gw;
        // Ring position of the up neighbour.  (A cell of the first row reads a
        // word that stays 0 until the cell 5 groups below its place is
        // decided.)
        int32_t rp = wrap((c - gw) % S.ring_n, S.ring_n);
        uint32_t ev;
        do {
            static_for<0, kSlots>([&](auto slot) __attribute__((always_inline)) {
                constexpr int s = decltype(slot)::value;
                uint32_t up[kPrepCells];
                bool first[kPrepCells];
#pragma unroll
                for (int k = 0; k < kPrepCells; ++k) {
                    up[k] = 0u;
                    if (kUp == kUpPrep)
                        up[k] = S.ring[rp + k < S.ring_n ? rp + k : rp + k - S.ring_n];
                    first[k] = x + k == (k == 0 ? 0 : gw);  // (x < gw)
                }
                prep_cells(q[s], c, cells, up, first, P, S, S.rows + s * kSlotWords, v * kPrepCells,
                           stage, lane);
                load_rows(job, c + kSlots * kGroup, cells, lane, q[s]);
                c += kGroup;
                x = kUp == kUpPrep ? (x + kGroup < gw ? x + kGroup : x + kGroup - gw)
                                   : (x + kGroup) % gw;
                rp += kGroup;
                rp = rp < S.ring_n ? rp : rp - S.ring_n;
                period_end(true);
            });
            ev = read_event(S, cycle);
        } while (!ev && ++cycle < cap);
        ++cycle;
        if (ev == kDone || cycle >= cap) return;
        start = (int32_t)ev - 1;
    }
}

// Winners from the ring to the grid, a cycle after the chain decided them,
// and the event words cleared two cycles ahead.
__device__ __forceinline__ void store_wave(const PlaceJob& job, const ChainShared& S, int lane) {
    const int32_t cells = job.grid_w * job.grid_h;
    const uint32_t cap = cycle_cap(cells);
    int32_t stored = 0, at = 0;  // cells stored, their ring position
    int32_t decided = 0;         // cells decided by the end of the last cycle
    bool fresh = true;           // the cycle is the first after a (re)start
    auto store_to = [&](int32_t end) {
        while (stored < end) {
            const int32_t k = min(end - stored, 64);
            int32_t i = at + lane;
            i = i < S.ring_n ? i : i - S.ring_n;
            if (lane < k) gstore(job.grid, stored + lane, entry_material(S.ring[i]));
            stored += k;
            at += k;
            at = at < S.ring_n ? at : at - S.ring_n;
        }
    };
    for (uint32_t cycle = 0; cycle < cap; ++cycle) {
        if (lane == 0) S.events[(cycle + 2) & (kEvents - 1)] = 0u;
        period_end(true);
        // (a period later: the chain's last ring write of the cycle before has
        // landed, see chain_wave)
        store_to(decided);
        period_end(true);
        period_end(true);
        const uint32_t ev = read_event(S, cycle);
        if (ev == kDone) break;
        decided = ev ? (int32_t)ev - 1 : decided + (fresh ? 1 : kSlots) * kGroup;
        fresh = ev != 0;
    }
    store_to(cells);
}

// ------------------------------------------------------------------ chain
// Index of the lowest set bit of a uniform mask, -1 when it is empty: the
// scalar find-first-one as is (the generic form adds a separate zero test).
__device__ __forceinline__ int32_t first_lane(uint64_t m) {
    // (m is uniform; the read-first-lanes only pin it to scalar registers)
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)(m >> 32));
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)(uint32_t)m);
    const uint64_t ms = ((uint64_t)hi << 32) | lo;
    int32_t r;
    asm("s_ff1_i32_b64 %0, %1" : "=s"(r) : "s"(ms));
    // an asm result counts as per-lane; re-reading it marks it uniform
    return __builtin_amdgcn_readfirstlane(r);
}

__device__ __forceinline__ uint32_t uniform_u(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)v);
}

__device__ __forceinline__ uint32_t readlane_u(uint32_t v, int lane) {
    return (uint32_t)__builtin_amdgcn_readlane((int32_t)v, lane);
}

struct ChainStats {
    int32_t ban, near, resets;
};

// An estimate of adj_term within 2^-18 of it (relative): the hardware's
// square root and reciprocal.
__device__ __forceinline__ float adj_term_estimate(float4 p, float4 q) {
    const float dl = p.x - q.x, da = p.y - q.y, db = p.z - q.z;
    const float s = __builtin_fmaf(db, db, __builtin_fmaf(da, da, dl * dl));
    return __builtin_amdgcn_rcpf(__builtin_amdgcn_sqrtf(s) + 1.0f);
}

// What a cell's candidates are scored against: Up then Left (Down and Right
// are still empty in raster order).
struct Neighbours {
    bool has_up, has_left;
    float4 up, left;
};
__device__ __forceinline__ float exact_score(float d, float4 lab, const Neighbours& nb, float weight) {
    float p = 0.0f;
    if (nb.has_up) p += adj_term(lab, nb.up);
    if (nb.has_left) p += adj_term(lab, nb.left);
    return d + p * weight;
}
__device__ __forceinline__ float score_estimate(float d, float4 lab, const Neighbours& nb,
                                                float weight) {
    const float tu = adj_term_estimate(lab, nb.up), tl = adj_term_estimate(lab, nb.left);
    return d + ((nb.has_up ? tu : 0.0f) + (nb.has_left ? tl : 0.0f)) * weight;
}
// A candidate whose estimate is above this cannot beat one estimated at e:
// both estimates are within 2^-17 of the scores, relative to the sum of
// distance and weight.
__device__ __forceinline__ float rival_bound(float e, float weight) {
    return e + (e + weight) * (1.0f / 16384.0f);
}

// Outcome of one evaluation of a whole row.
struct Decision {
    uint32_t w;      // the winner's entry id
    int32_t rank;
    int32_t stage;   // 0 scored scan, 1 fallback first-placeable, 2 nearest_one
    bool reset;
};

// (component by component: selecting between two float4 objects would keep
// both in memory)
__device__ __forceinline__ float4 select4(bool first, float4 a, float4 b) {
    return make_float4(first ? a.x : b.x, first ? a.y : b.y, first ? a.z : b.z, 0.0f);
}

// Material m's Lab, w = 0: a load of three words (a fourth that nobody reads
// is reused while it is still to be written, and the reuse waits for it).
__device__ __forceinline__ float4 load_lab(const PlaceJob& job, int32_t m) {
    typedef float f3 __attribute__((ext_vector_type(3)));
    const f3 v = *(const MH_GAS f3*)((const MH_GAS float4*)job.lab4 + m);
    return make_float4(v.x, v.y, v.z, 0.0f);
}

// The Labs of this lane's two candidates of a row (none: material 0's).
struct RowLabs {
    float4 l0, l1;
};
__device__ __forceinline__ RowLabs load_labs(const PlaceJob& job, const RawRow& row) {
    return RowLabs{load_lab(job, max((int32_t)(uint32_t)row.r0, 0)),
                   load_lab(job, max((int32_t)(uint32_t)row.r1, 0))};
}

// The evaluation of a cell from its whole row, and the usage-reset fallback
// (src/main.rs:385-475).  The first candidate wins at once if the others lie
// beyond the largest score it can have (two terms of at most 1); else
// estimates rule out all but the few that can win, and when those are
// several, exact scores decide.
__device__ __forceinline__ Decision decide_from_row(const PlaceJob& job, uint32_t* counts,
                                                    uint32_t limit, const RawRow& row,
                                                    const RowLabs& labs, uint32_t up, uint32_t left,
                                                    const Neighbours& nb, bool may_reset,
                                                    int lane) {
    const uint32_t kNone = 0xffffffffu;
    const uint32_t a0 = entry_id((int32_t)(uint32_t)row.r0), a1 = entry_id((int32_t)(uint32_t)row.r1);
    const float d0 = __uint_as_float((uint32_t)(row.r0 >> 32));
    const float d1 = __uint_as_float((uint32_t)(row.r1 >> 32));
    const uint64_t pl0 =
        lanes_ne((int32_t)a0, 0) & lanes_ne((int32_t)a0, (int32_t)up) & lanes_ne((int32_t)a0, (int32_t)left);
    const uint64_t pl1 =
        lanes_ne((int32_t)a1, 0) & lanes_ne((int32_t)a1, (int32_t)up) & lanes_ne((int32_t)a1, (int32_t)left);
    uint64_t b0 = pl0 & lanes_ult(counts[a0 >> 2], limit);
    uint64_t b1 = pl1 & lanes_ult(counts[a1 >> 2], limit);
    Decision r;
    r.stage = 0;
    r.reset = false;
    if (b0 | b1) {
        // (without a penalty the scores are the distances, which ascend)
        const float first = b0 ? readlane_f(d0, __ffsll((unsigned long long)b0) - 1)
                               : readlane_f(d1, __ffsll((unsigned long long)b1) - 1);
        const float reach = first + (job.weight > 0.0f ? 2.0f * job.weight : 0.0f);
        b0 &= wave_ballot(!(d0 > reach));
        b1 &= wave_ballot(!(d1 > reach));
        bool alone = __popcll(b0) + __popcll(b1) == 1;
        if (!alone && job.weight > 0.0f) {
            const float e0 = score_estimate(d0, labs.l0, nb, job.weight);
            const float e1 = score_estimate(d1, labs.l1, nb, job.weight);
            // keys: the scores' bits (no score is negative)
            const uint32_t k0 = lane_in(b0) ? __float_as_uint(e0) : kNone;
            const uint32_t k1 = lane_in(b1) ? __float_as_uint(e1) : kNone;
            const float far = rival_bound(__uint_as_float(wave_min_u32(k0 < k1 ? k0 : k1)), job.weight);
            b0 &= wave_ballot(!(e0 > far));
            b1 &= wave_ballot(!(e1 > far));
            alone = __popcll(b0) + __popcll(b1) == 1;
        }
        if (!alone && job.weight > 0.0f) {
            // one evaluation does for both candidates of a lane unless both are in
            const bool second = lane_in(b1 & ~b0);
            const float s =
                exact_score(second ? d1 : d0, select4(second, labs.l1, labs.l0), nb, job.weight);
            const uint32_t k0 = lane_in(b0) ? __float_as_uint(s) : kNone;
            uint32_t k1 = second ? __float_as_uint(s) : kNone;
            if (b0 & b1)
                k1 = lane_in(b1) ? __float_as_uint(exact_score(d1, labs.l1, nb, job.weight)) : kNone;
            const uint32_t score = wave_min_u32(k0 < k1 ? k0 : k1);
            b0 &= wave_ballot(k0 == score);
            b1 &= wave_ballot(k1 == score);
        }
    } else {
        // fallback_tile_selection: reset every count, first placeable, else nearest_one
        const uint32_t keep = packs(job) ? 0xffffu : 0u;
        if (may_reset)
            for (int32_t i = lane; i < job.n; i += 64) counts[1 + i] &= keep;
        r.reset = true;
        b0 = pl0;
        b1 = pl1;
        r.stage = (b0 | b1) ? 1 : 2;
        if (!(b0 | b1)) b0 = 1;
    }
    r.rank = b0 ? __ffsll((unsigned long long)b0) - 1 : 63 + __ffsll((unsigned long long)b1);
    r.w = r.rank < 64 ? readlane_u(a0, r.rank & 63) : readlane_u(a1, r.rank & 63);
    return r;
}

// The evaluation of a cell whose first usable entry may lose, from its list:
// a and d are this lane's entry and its distance, usable the mask of entries
// that can be taken, lab / nb_up / nb_left the Labs.  The first usable entry
// f wins unless another's estimated score comes within the estimates' error
// of f's; only then are those scores computed exactly.  False: the row beyond
// the list is needed.
__device__ __forceinline__ bool decide_from_list(const PlaceJob& job, uint32_t a, float d,
                                                 uint64_t usable, float4 lab, const Neighbours& nb,
                                                 uint32_t* w_out) {
    if (!usable) return false;
    const int32_t f = __ffsll((unsigned long long)usable) - 1;
    *w_out = readlane_u(a, f);
    if (!(job.weight > 0.0f)) return true;  // scores are the distances
    const float est = score_estimate(d, lab, nb, job.weight);
    const float far = rival_bound(readlane_f(est, f), job.weight);
    // the row may go on within reach
    if (!(readlane_f(d, 63) > far)) return false;
    const uint64_t field = usable & wave_ballot(!(est > far));  // f and its rivals
    if (field == (1ull << f)) return true;
    const bool in = lane_in(field | (1ull << f));
    const float s = exact_score(d, lab, nb, job.weight);
    const uint32_t key = in ? __float_as_uint(s) : 0xffffffffu;
    const uint32_t kmin = wave_min_u32(key);
    *w_out = readlane_u(a, __ffsll((unsigned long long)wave_ballot(in && key == kmin)) - 1);
    return true;
}

// What a chain knows of its grid.
struct ChainArgs {
    int32_t gw, cells;
    uint32_t limit, use;  // the usage limit and one use, in count words
    bool filtered;  // a reset invalidates the prepared lists
};

__device__ __forceinline__ ChainArgs chain_args(const PlaceJob& job) {
    ChainArgs A;
    A.gw = job.grid_w;
    A.cells = job.grid_w * job.grid_h;
    const uint32_t shift = packs(job) ? 16 : 0;
    A.limit = (uint32_t)job.max_usage << shift;
    A.use = 1u << shift;
    A.filtered = filters(job);
    return A;
}

// A flagged cell c < cells: its winner's entry id.  a: this lane's entry,
// left: the left neighbour (0 in a row's first cell), up_v: the up neighbour
// (the same in every lane), usable: the entries that can be taken (but in a
// row's first cell, which counts anew).  *reset: the counts were reset.
__device__ __forceinline__ uint32_t decide_flagged(const PlaceJob& job, const ChainShared& S,
                                                   const ChainArgs& A, int32_t c,
                                                   const uint32_t* dist, uint32_t a, uint32_t left,
                                                   uint32_t up_v, uint64_t usable, ChainStats& st,
                                                   bool* reset, int lane) {
    // every read in flight before the first is used (no entry, no neighbour:
    // material 0's Lab)
    const float d = reinterpret_cast<const float*>(dist)[lane];
    const int32_t ma = max(entry_material(a), 0), ml = max(entry_material(left), 0),
                  mu = max(entry_material(up_v), 0);
    float4 lab;
    Neighbours nb;
    if (S.labs) {
        lab = S.labs[ma];
        nb.left = S.labs[ml];
        nb.up = S.labs[mu];
    } else {
        lab = gload4(job.lab4, ma);
        nb.left = gload4(job.lab4, ml);
        nb.up = gload4(job.lab4, mu);
    }
    const uint32_t up = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)up_v);
    nb.has_up = up != 0u;
    nb.has_left = left != 0u;
    if (left == 0u)  // (the step banned the previous winner here)
        usable = lanes_ult(S.counts[a >> 2], A.limit) & lanes_ne((int32_t)a, (int32_t)up);
    uint32_t w;
    *reset = false;
    if (!decide_from_list(job, a, d, usable, lab, nb, &w)) {
        const RawRow row = load_row(job, c, A.cells, lane);
        const Decision r = decide_from_row(job, S.counts, A.limit, row, load_labs(job, row), up, left,
                                           nb, true, lane);
        w = r.w;
        if (r.reset) {
            ++st.resets;
            st.ban += r.stage == 1;
            st.near += r.stage == 2;
            if (job.stage && lane == 0) gstore(job.stage, c, (uint8_t)r.stage);
            *reset = true;
        }
    }
    return (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)w);
}

// The chain's event of this cycle (*period: the one it happened in), and the
// rest of the cycle.
__device__ __forceinline__ void leave_cycle(const ChainShared& S, uint32_t event, uint32_t* period,
                                            int lane) {
    const uint32_t cycle = *period / kSlots, rest = kSlots - (*period - cycle * kSlots);
    if (lane == 0) S.events[cycle & (kEvents - 1)] = event;
    for (uint32_t i = 0; i < rest; ++i) period_end(true);
    *period += rest;
}

// The chain.  Its step is written out in assembly: compiled
// from C++, the registers that carry entries and counts from cell to cell
// are copied at every point where the full evaluation can rejoin, and each
// copy waits for an LDS read that has a step or more left to land.
//
// The entries of three cells (with the flags) come in one read, into v[64:67]
// and v[68:71] in turn; cell c's entries without flags are in a[c mod 3], the
// counts of its entries in c[c mod 2], the winner in w[c mod 2]; u and fl are
// the masks of the entries below the limit and of the flagged ones.  The
// step of c
//   * takes the first entry in u that is not the previous winner; a flagged
//     one leaves the run (L_flagged);
//   * makes u and fl for c + 1, whose counts were read after the commit of
//     c - 1 (c's winner will be its left neighbour and banned, so that use
//     does not matter);
//   * commits: lane 0 adds a use, every other lane adds to its own scratch
//     word, so the commit has no branch on the lane; then reads c + 2's
//     counts (a wave's LDS operations are done in order: after the commit).
// A wave issues an instruction every 4 cycles, but a scalar instruction that
// follows a vector compare or lane read waits about 16 more, a branch takes
// 12 and an LDS instruction among vector ones 8 (measured); the order below
// is the best of some 300 measured, 88 cycles a step (128 for the plain one).
// The steps begin on a 256-byte boundary: 1-2% for their instruction fetch.
//
// Flags of an entry: kFlagged any of the others; kFirst the row's first
// cell, which has no left neighbour -- the step is right for it all the same
// unless the previous winner is on its list; kUnsafe as above.
//
// At the end of a group its winners go to the ring (lane i: cell i's), the
// row addresses move on and the waves meet.  This wave's LDS operations are
// not waited for there: its ring writes are read by others a period later
// at the earliest, when it has waited for reads that were issued after them.
//
// kUpChain: up and ban, further instructions that keep the last 64 winners in
// hist (cell c's in lane c mod 64, m0 = c) and take c + 1's up neighbour out
// of u for c + 1 (ban: the mask of its entries); 28 cycles more a step.  m0 is
// the compiler's (a reserved register, which a clobber list cannot name): it is
// put back on the way out.
//
// Entered with slot = 12 at cell g0, or after a full evaluation of the cell
// in `slot` at its commit; left at a flagged cell with everything landed.
// Wait states: a lane read's scalar result has two instructions before a
// vector instruction uses it.
#define MH_STEP(I, A, B, C, MB, MC, CB, CC, WN, READ, BAN, KEEP, UP)    \
    "L_dec" #I "_%=:\n"                                                 \
    BAN                                                                 \
    "s_andn2_b64 %[u], %[u], vcc\n"                                     \
    "s_ff1_i32_b64 %[f], %[u]\n"                                        \
    "s_bitcmp1_b64 %[fl], %[f]\n"                                       \
    "v_readlane_b32 %[w" #WN "], %[a" #A "], %[f]\n"                    \
    "s_cbranch_scc1 L_flagged" #I "_%=\n"                               \
    "L_adv" #I "_%=:\n"                                                 \
    "v_and_b32_e32 %[a" #C "], %[ids], " #MC "\n"                       \
    KEEP(WN)                                                            \
    "v_cmp_eq_u32_e32 vcc, %[w" #WN "], %[a" #B "]\n"                   \
    "s_waitcnt lgkmcnt(0)\n"                                            \
    "v_cmp_gt_i32_e64 %[fl], 0, " #MB "\n"                              \
    READ                                                                \
    "v_cmp_gt_u32_e64 %[u], %[lim], %[c" #CB "]\n"                      \
    UP(B)                                                               \
    "v_mad_u32_u24 %[t], %[w" #WN "], %[mul], %[port]\n"                \
    "ds_add_u32 %[t], %[one] offset:%[counts]\n"                        \
    "ds_read_b32 %[c" #CC "], %[a" #C "] offset:%[counts]\n"            \
    "v_writelane_b32 %[wins], %[w" #WN "], " #I "\n"
#define MH_NO(X) ""
#define MH_BAN "s_andn2_b64 %[u], %[u], %[ban]\n"
#define MH_KEEP(WN)                                                     \
    "v_writelane_b32 %[hist], %[w" #WN "], m0\n"                        \
    "s_add_u32 m0, m0, 1\n"                                             \
    "s_sub_u32 %[up], m0, %[gw]\n"                                      \
    "v_readlane_b32 %[up], %[hist], %[up]\n"
#define MH_TAKE_M0 "s_mov_b32 %[m0s], m0\ns_mov_b32 m0, %[cell]\n"
#define MH_GIVE_M0 "s_mov_b32 m0, %[m0s]\n"
#define MH_UP(B) "v_cmp_eq_u32_e64 %[ban], %[up], %[a" #B "]\n"
#define MH_READ(Q, ROW, T) "ds_read_b128 " Q ", %[" #ROW "] offset:" #T "*1024\n"
// A flagged cell (its entry is read again: the registers may hold a later
// cell's) that is only its row's first, with the previous winner not on its
// list, goes on.  Otherwise out: t the cell's entries, f the flagged one's
// word, wp the previous winner.
#define MH_FLAGGED(I, A, T, K, WP)                                      \
    "L_flagged" #I "_%=:\n"                                             \
    "ds_read_b32 %[t], %[rc] offset:" #T "*1024+4*" #K "\n"             \
    "v_cmp_eq_u32_e32 vcc, %[w" #WP "], %[a" #A "]\n"                   \
    "s_mov_b32 %[slot], " #I "\n"                                       \
    "s_mov_b32 %[wp], %[w" #WP "]\n"                                    \
    "s_waitcnt lgkmcnt(0)\n"                                            \
    "v_readlane_b32 %[f], %[t], %[f]\n"                                 \
    "v_mov_b32_e32 %[t], %[a" #A "]\n"                                  \
    "s_bitcmp1_b32 %[f], %[unsafe]\n"                                   \
    "s_cbranch_scc1 L_exit_%=\n"                                        \
    "s_cbranch_vccz L_adv" #I "_%=\n"                                   \
    "s_branch L_exit_%=\n"
// Enters the commit of one of three cells, `slot`.
#define MH_ENTER(I0, I1, I2)                \
    "s_cmp_eq_u32 %[slot], " #I0 "\n"       \
    "s_cbranch_scc1 L_adv" #I0 "_%=\n"      \
    "s_cmp_eq_u32 %[slot], " #I1 "\n"       \
    "s_cbranch_scc1 L_adv" #I1 "_%=\n"      \
    "s_branch L_adv" #I2 "_%=\n"

// (cell, a of c, c + 1, c + 2, entries of c + 1, c + 2, their counts, w)
#define MH_RUN(BAN, KEEP, UP, TAKE, GIVE)                                                       \
    asm volatile(                                                                               \
        TAKE                                                                                    \
        "s_cmp_eq_u32 %[slot], 12\n"                                                            \
        "v_cmp_eq_u32_e32 vcc, %[w1], %[a0]\n"                                                  \
        "s_cbranch_scc1 L_dec0_%=\n"                                                            \
        "s_cmp_lt_u32 %[slot], 6\n"                                                             \
        "s_cbranch_scc1 L_low_%=\n"                                                             \
        "s_cmp_lt_u32 %[slot], 9\n"                                                             \
        "s_cbranch_scc1 L_in6_%=\n"                                                             \
        MH_ENTER(9, 10, 11)                                                                     \
        "L_in6_%=:\n"                                                                           \
        MH_ENTER(6, 7, 8)                                                                       \
        "L_low_%=:\n"                                                                           \
        "s_cmp_lt_u32 %[slot], 3\n"                                                             \
        "s_cbranch_scc1 L_in0_%=\n"                                                             \
        MH_ENTER(3, 4, 5)                                                                       \
        "L_in0_%=:\n"                                                                           \
        MH_ENTER(0, 1, 2)                                                                       \
        ".p2align 8\n"                                                                          \
        MH_STEP(0, 0, 1, 2, v65, v66, 1, 0, 0, "", BAN, KEEP, UP)                               \
        MH_STEP(1, 1, 2, 0, v66, v68, 0, 1, 1, MH_READ("v[64:67]", rc, 2), BAN, KEEP, UP)       \
        MH_STEP(2, 2, 0, 1, v68, v69, 1, 0, 0, "", BAN, KEEP, UP)                               \
        MH_STEP(3, 0, 1, 2, v69, v70, 0, 1, 1, "", BAN, KEEP, UP)                               \
        MH_STEP(4, 1, 2, 0, v70, v64, 1, 0, 0, MH_READ("v[68:71]", rc, 3), BAN, KEEP, UP)       \
        MH_STEP(5, 2, 0, 1, v64, v65, 0, 1, 1, "", BAN, KEEP, UP)                               \
        MH_STEP(6, 0, 1, 2, v65, v66, 1, 0, 0, "", BAN, KEEP, UP)                               \
        MH_STEP(7, 1, 2, 0, v66, v68, 0, 1, 1, MH_READ("v[64:67]", rn, 0), BAN, KEEP, UP)       \
        MH_STEP(8, 2, 0, 1, v68, v69, 1, 0, 0, "", BAN, KEEP, UP)                               \
        MH_STEP(9, 0, 1, 2, v69, v70, 0, 1, 1, "", BAN, KEEP, UP)                               \
        MH_STEP(10, 1, 2, 0, v70, v64, 1, 0, 0, MH_READ("v[68:71]", rn, 1), BAN, KEEP, UP)      \
        MH_STEP(11, 2, 0, 1, v64, v65, 0, 1, 1, "", BAN, KEEP, UP)                              \
        "s_mov_b64 exec, 0xfff\n"                                                               \
        "ds_write_b32 %[ring], %[wins]\n"                                                       \
        "s_mov_b64 exec, -1\n"                                                                  \
        "v_add_u32_e32 %[ring], 48, %[ring]\n"                                                  \
        "v_cmp_le_u32_e32 vcc, %[rend], %[ring]\n"                                              \
        "v_subrev_u32_e32 %[t], %[rlen], %[ring]\n"                                             \
        "s_add_u32 %[g0], %[g0], 12\n"                                                          \
        "s_add_u32 %[per], %[per], 1\n"                                                         \
        "v_cndmask_b32_e32 %[ring], %[ring], %[t], vcc\n"                                       \
        "v_mov_b32_e32 %[rc], %[rn]\n"                                                          \
        "s_add_u32 %[so], %[so], %[slotb]\n"                                                    \
        "s_cmp_eq_u32 %[so], 3*%[slotb]\n"                                                      \
        "s_cselect_b32 %[so], 0, %[so]\n"                                                       \
        "v_add_u32_e32 %[rn], %[so], %[row0]\n"                                                 \
        "v_cmp_eq_u32_e32 vcc, %[w1], %[a0]\n"                                                  \
        "s_barrier\n"                                                                           \
        "s_branch L_dec0_%=\n"                                                                  \
        MH_FLAGGED(0, 0, 0, 0, 1) MH_FLAGGED(1, 1, 0, 1, 0) MH_FLAGGED(2, 2, 0, 2, 1)           \
        MH_FLAGGED(3, 0, 1, 0, 0) MH_FLAGGED(4, 1, 1, 1, 1) MH_FLAGGED(5, 2, 1, 2, 0)           \
        MH_FLAGGED(6, 0, 2, 0, 1) MH_FLAGGED(7, 1, 2, 1, 0) MH_FLAGGED(8, 2, 2, 2, 1)           \
        MH_FLAGGED(9, 0, 3, 0, 0) MH_FLAGGED(10, 1, 3, 1, 1) MH_FLAGGED(11, 2, 3, 2, 0)         \
        "L_exit_%=:\n"                                                                          \
        GIVE                                                                                    \
        "s_waitcnt lgkmcnt(0)\n"                                                                \
        : "+{v[64:67]}"(q0), "+{v[68:71]}"(q1), [a0] "+v"(a0), [a1] "+v"(a1), [a2] "+v"(a2),    \
          [c0] "+v"(c0), [c1] "+v"(c1), [wins] "+v"(wins), [rc] "+v"(rows_c),                   \
          [rn] "+v"(rows_n), [ring] "+v"(ring_w), [t] "=&v"(t), [u] "+s"(u), [fl] "+s"(fl),     \
          [w0] "+s"(w0), [w1] "+s"(w1), [wp] "=&s"(prev), [f] "=&s"(f),                         \
          [slot] "+s"(slot), [g0] "+s"(g0),                                                     \
          [per] "+s"(period), [so] "+s"(so), [hist] "+v"(hist), [up] "=&s"(up), [ban] "+s"(ban), \
          [m0s] "=&s"(m0_saved)                                                                 \
        : [mul] "v"(mul), [port] "v"(port), [one] "v"(one), [row0] "v"(row0),                   \
          [lim] "s"(A.limit), [rend] "s"(ring_end), [rlen] "s"(ring_b),                         \
          [ids] "s"(kEntryId), [counts] "n"(kCountBytes), [slotb] "n"(kSlotBytes),              \
          [unsafe] "n"(kUnsafeBit), [cell] "s"(cell), [gw] "s"(A.gw)                            \
        : "memory", "vcc", "scc")

template <int kUp>
__device__ __forceinline__ ChainStats chain_wave(const PlaceJob& job, const ChainShared& S, int lane) {
    static_assert(kGroup == 12 && kSlots == 3, "the steps below");
    typedef __attribute__((address_space(3))) uint32_t lds_u32;
    auto lds = [](uint32_t* p) { return (uint32_t)(uintptr_t)(lds_u32*)p; };
    ChainStats st{0, 0, 0};
    const ChainArgs A = chain_args(job);
    constexpr uint32_t kSlotBytes = kSlotWords * 4;
    constexpr uint32_t kCountBytes = kCountsAt * 4;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    // (the kernel's LDS starts at address 0)
    const uint32_t mul = lane == 0 ? 1u : 0u;
    const uint32_t port = lane == 0 ? 0u : lds(S.scratch + lane) - kCountBytes;
    const uint32_t one = A.use;
    const uint32_t row0 = lds(S.rows + 4 * lane);   // this lane's entries of the first slot
    const uint32_t ring_end = lds(S.ring + S.ring_n), ring_b = 4u * (uint32_t)S.ring_n;
    uint32_t ring_w = lds(S.ring + lane);           // where the group's winner `lane` goes
    uint32_t period = 0, w0 = 0, w1 = 0, wins = 0, hist = 0;
    int32_t g0 = 0, cell = 0;                       // cell: the next to decide or commit
    bool running = true;
    while (running) {
        // (re)start at g0: the first two groups are prepared
        period_end(true);
        period_end(true);
        period += 2;
        uint32_t so = kSlotBytes;                   // LDS offset of the next group's slot
        uint32_t rows_c = row0, rows_n = row0 + so;  // this lane's entries of both groups
        u32x4 q0 = *reinterpret_cast<const u32x4*>(S.rows + 4 * lane);
        u32x4 q1 = *reinterpret_cast<const u32x4*>(S.rows + 256 + 4 * lane);
        uint32_t a0 = q0.x & kEntryId, a1 = q0.y & kEntryId, a2 = 0;
        uint32_t c0 = 0, c1 = S.counts[a1 >> 2];
        uint64_t u = lanes_ult(S.counts[a0 >> 2], A.limit);
        uint64_t fl = __builtin_amdgcn_sicmp((int32_t)q0.x, 0, 40);  // < 0
        uint64_t ban = 0;
        if (kUp == kUpChain) ban = lanes_eq((int32_t)a0, (int32_t)readlane_u(hist, (cell - A.gw) & 63));
        int32_t slot = kGroup;
        bool restart = false;
        while (!restart) {
            uint32_t t, prev, up, m0_saved;
            int32_t f;
            if constexpr (kUp == kUpPrep)
                MH_RUN("", MH_NO, MH_NO, "", "");
            else
                MH_RUN(MH_BAN, MH_KEEP, MH_UP, MH_TAKE_M0, MH_GIVE_M0);
            slot = __builtin_amdgcn_readfirstlane(slot);
            f = __builtin_amdgcn_readfirstlane(f);  // the flagged entry
            g0 = __builtin_amdgcn_readfirstlane(g0);
            period = uniform_u(period);
            so = uniform_u(so);
            u = (uint64_t)uniform_u((uint32_t)(u >> 32)) << 32 | uniform_u((uint32_t)u);
            const int32_t c = g0 + slot;
            cell = c;
            uint32_t decided = (uint32_t)slot;  // cells of the group decided
            if (c >= A.cells) {
                running = false;
            } else {
                const int32_t slot_c = so == 0 ? 2 : so == kSlotBytes ? 0 : 1;
                if (kUp == kUpChain) {
                    up = readlane_u(hist, (c - A.gw) & 63);
                } else {
                    // (cell g0's ring word is lane 0's ring_w)
                    const int32_t i = (int32_t)((uniform_u(ring_w) - lds(S.ring)) >> 2) + slot - A.gw;
                    up = S.ring[wrap(i, S.ring_n)];
                }
                bool reset;
                const uint32_t w =
                    decide_flagged(job, S, A, c, S.rows + slot_c * kSlotWords + dist_word(slot, 0), t,
                                   (f & kFirst) ? 0u : uniform_u(prev), up, u, st, &reset, lane);
                if (slot & 1)
                    w1 = w;
                else
                    w0 = w;
                if (reset) {
                    if (A.filtered) {
                        // commit here; the lists prepared before the reset are void
                        restart = true;
                        if (lane == 0) S.counts[w >> 2] += A.use;
                        wins = lane == slot ? w : wins;
                        hist = lane == (c & 63) ? w : hist;
                        cell = c + 1;
                        // (re)started at cell 0 of a group: its previous winner is w[1]
                        w1 = w;
                        ++decided;
                    } else {
                        // the next cell's counts were read before the reset
                        const int32_t k = slot % 3;
                        const uint32_t an = k == 0 ? a1 : k == 1 ? a2 : a0;
                        const uint32_t cn = S.counts[an >> 2];
                        if (slot & 1)
                            c0 = cn;
                        else
                            c1 = cn;
                    }
                }
            }
            if (restart || !running) {
                if ((uint32_t)lane < decided) *(lds_u32*)(uintptr_t)ring_w = wins;
                ring_w += 4u * decided;
                ring_w = ring_w < ring_end ? ring_w : ring_w - ring_b;
                g0 += (int32_t)decided;
                leave_cycle(S, running ? (uint32_t)g0 + 1u : kDone, &period, lane);
                if (!running) break;
            }
        }
    }
    return st;
}
#undef MH_STEP
#undef MH_READ
#undef MH_FLAGGED
#undef MH_ENTER
#undef MH_RUN
#undef MH_NO
#undef MH_BAN
#undef MH_KEEP
#undef MH_UP
#undef MH_TAKE_M0
#undef MH_GIVE_M0

// kRasterPlain: one cell at a time from the whole row, the row above in
// S.ring.  For grids of one or two columns, where the lists would be prepared
// after their cells are decided, and for libraries whose counts leave LDS no
// place for lists.  Bound by the latency of a scored row; the next cell's Labs and
// the rows of the four after this one are in flight meanwhile (four cells an
// iteration and no branch around the loads, so that the compiler's waits are
// for the Labs alone: cells past the grid are evaluated and dropped; one column
// is compiled by itself, as a choice of the up neighbour's Lab at run time
// waits for it a cell early).  Every candidate scored 0.67 us a cell of 36,000
// materials, the first alone where it can be 0.57, without that wait 0.56; GUI
// score 0.69, 0.65, 0.62.
template <bool kOneColumn>
__device__ __forceinline__ ChainStats raster_plain(const PlaceJob& job, const ChainShared& S, int lane) {
    constexpr int kRows = 4;
    ChainStats st{0, 0, 0};
    const ChainArgs A = chain_args(job);
    Neighbours nb{};
    uint32_t w = 0, won = 0;
    RawRow row[kRows];
    RowLabs labs[2];
    float4 lab_up[2] = {nb.up, nb.up};
#pragma unroll
    for (int k = 0; k < kRows; ++k) row[k] = load_row(job, k, A.cells, lane);
    labs[0] = load_labs(job, row[0]);
    int32_t x = 0;
    for (int32_t c4 = 0; c4 < A.cells; c4 += kRows) {
        static_for<0, kRows>([&](auto slot) __attribute__((always_inline)) {
            constexpr int k = decltype(slot)::value;
            const int32_t c = c4 + k;
            const bool valid = c < A.cells;
            const int32_t x1 = x + 1 < A.gw ? x + 1 : 0;
            const uint32_t up = uniform_u(S.ring[x]), left = x ? w : 0u;
            const RawRow cur = row[k];
            labs[(k + 1) & 1] = load_labs(job, row[(k + 1) % kRows]);
            lab_up[(k + 1) & 1] = load_lab(job, max(entry_material(S.ring[x1]), 0));
            row[k] = load_row(job, c + kRows, A.cells, lane);
            nb.has_up = up != 0u;
            nb.has_left = left != 0u;
            nb.up = kOneColumn ? nb.left : lab_up[k & 1];  // (one column: the previous winner)
            const Decision r = decide_from_row(job, S.counts, valid ? A.limit : kGuard, cur,
                                               labs[k & 1], up, left, nb, valid, lane);
            w = r.w;
            const float4 lab = select4(r.rank < 64, labs[k & 1].l0, labs[k & 1].l1);
            const int32_t from = r.rank & 63;
            nb.left = make_float4(readlane_f(lab.x, from), readlane_f(lab.y, from),
                                  readlane_f(lab.z, from), 0);
            if (valid) {
                st.resets += r.reset;
                st.ban += r.stage == 1;
                st.near += r.stage == 2;
                if (lane == 0) {
                    S.counts[w >> 2] += A.use;
                    S.ring[x] = w;
                    if (r.reset && job.stage) gstore(job.stage, c, (uint8_t)r.stage);
                }
            }
            asm volatile("" ::: "memory");
            x = x1;
            won = lane == (c & 63) ? w : won;  // (stored 64 cells at a time)
        });
        if ((c4 & 63) == 64 - kRows || c4 + kRows >= A.cells) {
            const int32_t i = (c4 & ~63) + lane;
            if (i < A.cells && i < c4 + kRows) gstore(job.grid, i, entry_material(won));
        }
    }
    return st;
}

__global__ __launch_bounds__(kChainThreads) void place_raster_kernel(
    PlaceJob single, const PlaceJob* __restrict__ jobs) {
    extern __shared__ __align__(16) uint32_t smr[];
    const PlaceJob job = uniform_copy(jobs ? jobs[blockIdx.x] : single);
    const int tid = threadIdx.x, lane = tid & 63;
    const int32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int32_t gw = job.grid_w, n = job.n;
    const int32_t cells = gw * job.grid_h;
    if (n == 0) {  // src/main.rs:342-345: no tiles, every cell stays empty
        for (int32_t i = tid; i < cells; i += kChainThreads) gstore(job.grid, i, kEmpty);
        if (tid == 0 && job.stats) {
            for (int i = 0; i < 5; ++i) gstore(job.stats, i, 0);
            gstore(job.stats, 5, cells);
        }
        return;
    }
    ChainShared S;
    S.events = smr;
    S.counts = smr + kCountsAt;
    S.scratch = smr + scratch_at(n);
    S.ring = smr + ring_at(n);
    S.ring_n = job.form == kRasterPlain ? gw : ring_words(gw);
    S.rows = smr + rows_at(gw, n);
    S.stage = S.rows + kSlots * kSlotWords;
    S.labs = job.form == kRasterLabs ? reinterpret_cast<float4*>(smr + labs_at(gw, n)) : nullptr;
    if (S.labs)
        for (int32_t i = tid; i < n; i += kChainThreads) S.labs[i] = gload4(job.lab4, i);
    const bool packed = packs(job);
    const bool terms = packed && job.form != kRasterPlain;
    for (int32_t i = tid; i < n; i += kChainThreads)
        S.counts[1 + i] = terms ? bf16_up(gload4(job.lab4, i).w) >> 16
                                : (job.zero_usage ? 0u : gload(job.usage, i));
    for (int32_t i = tid; i < S.ring_n; i += kChainThreads) S.ring[i] = 0u;
    if (tid < kEvents) S.events[tid] = 0u;
    if (tid == 0) S.counts[0] = kGuard;
    // every cell's stage is 0 but for those whose decision resets the counts
    if (job.stage)
        for (int32_t i = tid; i < cells; i += kChainThreads) gstore(job.stage, i, (uint8_t)0);
    __syncthreads();

    if (wave == 0) {
        ChainStats st;
        if (job.form == kRasterPlain && gw == 1)
            st = raster_plain<true>(job, S, lane);
        else if (job.form == kRasterPlain)
            st = raster_plain<false>(job, S, lane);
        else if (gw < kUpPrepColumns)
            st = chain_wave<kUpChain>(job, S, lane);
        else
            st = chain_wave<kUpPrep>(job, S, lane);
        if (lane == 0 && job.stats) {
            gstore(job.stats, 0, cells);
            gstore(job.stats, 1, cells - st.ban - st.near);
            gstore(job.stats, 2, st.ban);
            gstore(job.stats, 3, st.near);
            gstore(job.stats, 4, st.resets);
            gstore(job.stats, 5, 0);
        }
    } else if (job.form != kRasterPlain) {
        const int32_t v = wave < kStoreWave ? wave - 1 : wave - 2;
        if (wave == kStoreWave)
            store_wave(job, S, lane);
        else if (gw < kUpPrepColumns)
            prep_waves<kUpChain>(job, S, v, lane);
        else
            prep_waves<kUpPrep>(job, S, v, lane);
    }
    __syncthreads();
    for (int32_t i = tid; i < n; i += kChainThreads)
        gstore(job.usage, i, S.counts[1 + i] >> (packed ? 16 : 0));
}

// What a raster run's cells won with, from the grid it left (and, for the
// scores, its stages): a cell's up and left neighbours are those it was
// decided against.  A wave to a cell, which finds the winner in its row.  The
// chain itself keeps only the stages of resets: with distances and scores it
// would score every cell (80 x 60 cells: 4.2 ms, the chain 0.27).
__global__ __launch_bounds__(256) void place_outputs_kernel(PlaceJob job) {
    const int lane = threadIdx.x & 63;
    const int32_t c = __builtin_amdgcn_readfirstlane((int32_t)(blockIdx.x * 4 + (threadIdx.x >> 6)));
    const int32_t gw = job.grid_w, cells = gw * job.grid_h;
    if (c >= cells) return;
    const RawRow row = load_row(job, c, cells, lane);
    const int32_t x = c % gw, m = gload(job.grid, c);
    const bool second = (int32_t)(uint32_t)row.r1 == m;
    const uint64_t at = wave_ballot((int32_t)(uint32_t)row.r0 == m || second);
    if (!at) return;  // (a placed tile is on its cell's row)
    const float d = readlane_f(__uint_as_float((uint32_t)((second ? row.r1 : row.r0) >> 32)),
                               __ffsll((unsigned long long)at) - 1);
    if (lane != 0) return;
    if (job.dist) gstore(job.dist, c, d);
    if (!job.score) return;
    float score = d;
    if (job.weight > 0.0f && gload(job.stage, c) == 0) {
        Neighbours nb{};
        nb.has_up = c >= gw;
        nb.has_left = x > 0;
        if (nb.has_up) nb.up = load_lab(job, gload(job.grid, c - gw));
        if (nb.has_left) nb.left = load_lab(job, gload(job.grid, c - 1));
        score = exact_score(d, load_lab(job, m), nb, job.weight);
    }
    gstore(job.score, c, score);
}

void launch_place_outputs(const PlaceJob& job, hipStream_t stream) {
    if (job.n <= 0 || !(job.dist || job.score)) return;
    hipLaunchKernelGGL(place_outputs_kernel, dim3((job.grid_w * job.grid_h + 3) / 4), dim3(256), 0,
                       stream, job);
}

size_t place_lds_bytes(int32_t cells, int32_t n) {
    return sizeof(int32_t) * ((size_t)cells + (size_t)n);
}

size_t place_raster_lds_bytes(int32_t grid_w, int32_t n, int32_t form) {
    const size_t words = form == kRasterPlain ? (size_t)ring_at(n) + (size_t)grid_w
                                              : (size_t)labs_at(grid_w, n);
    return sizeof(uint32_t) * (words + (form == kRasterLabs ? 4 * (size_t)n : 0));
}

// Where each form stands: the lists take 28 KB and 4 bytes a material (to
// about 33,800 materials), the Labs 16 bytes a material more.  A flagged
// cell's Labs come from LDS in 0.4 us, from memory in 0.7-1 us.  Without room
// for the lists (33,800 to 40,700 materials) a cell costs 0.56 us plain, as
// one wave that read ahead in registers did.
//
// Without the materials' largest terms a list's entries would all look safe,
// so such a library's runs are plain; lists_taken says which libraries need
// the terms (33,828 to 33,847 materials: in grids of 48 to 67 columns only).
bool lists_taken(int32_t n, size_t max_lds) {
    return place_raster_lds_bytes(kLeastRingColumns, n, kRasterLists) <= max_lds;
}
int32_t raster_form(int32_t grid_w, int32_t n, bool labs, bool terms, size_t max_lds) {
    const bool plain = grid_w < 3 || !terms;
    for (int32_t form = plain ? kRasterPlain : labs ? kRasterLabs : kRasterLists; form >= 0; --form)
        if (place_raster_lds_bytes(grid_w, n, form) <= max_lds) return form;
    return -1;
}

void launch_place_single(const PlaceJob& job, bool raster, size_t lds_bytes, hipStream_t stream) {
    const PlaceJob* none = nullptr;
    if (raster)
        hipLaunchKernelGGL(place_raster_kernel, dim3(1), dim3(kChainThreads), lds_bytes, stream, job,
                           none);
    else if (lds_bytes > 0)
        hipLaunchKernelGGL(place_chain_kernel<false>, dim3(1), dim3(64), lds_bytes, stream, job, none);
    else
        hipLaunchKernelGGL(place_chain_kernel<true>, dim3(1), dim3(64), 0, stream, job, none);
}

void launch_place_batch(const PlaceJob* d_jobs, int32_t n_jobs, bool raster, size_t lds_bytes,
                        hipStream_t stream) {
    if (n_jobs <= 0) return;
    PlaceJob unused{};
    if (raster)
        hipLaunchKernelGGL(place_raster_kernel, dim3(n_jobs), dim3(kChainThreads), lds_bytes, stream,
                           unused, d_jobs);
    else if (lds_bytes > 0)
        hipLaunchKernelGGL(place_chain_kernel<false>, dim3(n_jobs), dim3(64), lds_bytes, stream,
                           unused, d_jobs);
    else
        hipLaunchKernelGGL(place_chain_kernel<true>, dim3(n_jobs), dim3(64), 0, stream, unused,
                           d_jobs);
}

hipError_t place_configure(int max_lds) {
    const void* kernels[] = {
        reinterpret_cast<const void*>(&place_chain_kernel<false>),
        reinterpret_cast<const void*>(&place_raster_kernel),
    };
    for (const void* k : kernels) {
        const hipError_t e = raise_dynamic_lds(k, max_lds);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace mh
