// Device primitives for gfx950 (CDNA4, wave64): lane/ballot helpers,
// wave-aggregated queue appends and a bounded, two-level grid barrier for
// cooperatively launched persistent kernels.
//
// These replace the reference's cub warp primitives (ShuffleIndex<32>,
// LaneId, LaneMaskLt, WarpReduce) and cub::GridBarrier
// (include/groute/device/cta_scheduler_hybrid.cuh:150-253,
// include/groute/device/queue.cuh:60-114,
// include/framework/algo_variants.cuh:353-355). Ballots here are 64-bit.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sg {

constexpr int kWave = 64;

__device__ __forceinline__ int lane() { return (int)__lane_id(); }

// Number of lanes below this one whose bit is set in `mask`.
__device__ __forceinline__ int rank_in(uint64_t mask)
{
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                          __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

__device__ __forceinline__ uint64_t ballot(bool p) { return __ballot(p); }

__device__ __forceinline__ int first_lane(uint64_t mask) { return __ffsll((unsigned long long)mask) - 1; }

template <typename T>
__device__ __forceinline__ T shfl(T v, int src) { return __shfl(v, src, kWave); }

// The value lane l (the same in every lane) holds, in every lane, without a
// trip through LDS: v_readlane instead of ds_bpermute's ~60 clocks. Wave-convergent.
template <typename T>
__device__ __forceinline__ T lane_value(T v, int l)
{
    static_assert(sizeof(T) % 4 == 0, "whole registers");
    constexpr int N = (int)(sizeof(T) / 4);
    int w[N];
    __builtin_memcpy(w, &v, sizeof(T));
    const int at = __builtin_amdgcn_readfirstlane(l);
#pragma unroll
    for (int i = 0; i < N; i++) w[i] = __builtin_amdgcn_readlane(w[i], at);
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
}

// Data-parallel-primitive controls: a move across lanes inside a vector
// instruction (a few clocks) where a shuffle goes through LDS (~60 clocks).
constexpr int kDppQuad1 = 0xB1;        // lanes of a pair trade places
constexpr int kDppQuad2 = 0x4E;        // pairs of a quad trade places
constexpr int kDppRowShr = 0x110;      // + k: lane i of a row of 16 takes lane i - k
constexpr int kDppRowRor = 0x120;      // + k: the same, from the row's end on
constexpr int kDppWaveShl1 = 0x130;    // lane i takes lane i + 1
constexpr int kDppWaveShr1 = 0x138;    // lane i takes lane i - 1
constexpr int kDppHalfMirror = 0x141;  // lane i of 8 takes lane 7 - i
constexpr int kDppRowBcast15 = 0x142;  // a row takes the last lane of the row before it
constexpr int kDppRowBcast31 = 0x143;  // rows 2 and 3 take lane 31

// `v` of the lane the control names; lanes it names none for, and rows outside
// kRows, take `none`.
template <int kCtrl, int kRows = 0xf, typename T>
__device__ __forceinline__ T dpp(T none, T v)
{
    static_assert(sizeof(T) % 4 == 0, "whole registers");
    constexpr int N = (int)(sizeof(T) / 4);
    int w[N], o[N];
    __builtin_memcpy(w, &v, sizeof(T));
    __builtin_memcpy(o, &none, sizeof(T));
#pragma unroll
    for (int i = 0; i < N; i++) w[i] = __builtin_amdgcn_update_dpp(o[i], w[i], kCtrl, kRows, 0xf, false);
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
}

// Inclusive scan across the wave with op(lower lanes, higher lanes) and its
// neutral value: four steps inside the rows of 16 lanes, then each odd row
// takes its lower neighbour's total, then the upper half takes lane 31's.
// A scan is a serial chain that every scheduling step and counter of a round
// waits for. By six shuffles each waited for in turn, it had cost 5-28 % of
// whole calls: RMAT-12 BFS 62.9 us with them and 56.1 without, RMAT-22 BFS 182
// and 173, RMAT-21 PageRank 2871 and 2654, 64-source BC on RMAT-16 2844 and 2224.
template <typename T, typename Op>
__device__ __forceinline__ T wave_scan(T x, T none, Op op)
{
    x = op(dpp<kDppRowShr + 1>(none, x), x);
    x = op(dpp<kDppRowShr + 2>(none, x), x);
    x = op(dpp<kDppRowShr + 4>(none, x), x);
    x = op(dpp<kDppRowShr + 8>(none, x), x);
    x = op(dpp<kDppRowBcast15, 0xa>(none, x), x);
    x = op(dpp<kDppRowBcast31, 0xc>(none, x), x);
    return x;
}

// The same within runs of adjacent lanes of one `key` (any value but ~0).
template <typename T, typename Op>
__device__ __forceinline__ T wave_seg_scan(T x, uint32_t key, Op op)
{
    auto step = [&](const T &y, uint32_t ky) {
        if (ky == key) x = op(y, x);
    };
    step(dpp<kDppRowShr + 1>(x, x), dpp<kDppRowShr + 1>(~0u, key));
    step(dpp<kDppRowShr + 2>(x, x), dpp<kDppRowShr + 2>(~0u, key));
    step(dpp<kDppRowShr + 4>(x, x), dpp<kDppRowShr + 4>(~0u, key));
    step(dpp<kDppRowShr + 8>(x, x), dpp<kDppRowShr + 8>(~0u, key));
    step(dpp<kDppRowBcast15, 0xa>(x, x), dpp<kDppRowBcast15, 0xa>(~0u, key));
    step(dpp<kDppRowBcast31, 0xc>(x, x), dpp<kDppRowBcast31, 0xc>(~0u, key));
    return x;
}

// A reduction over the wave, in every lane (the scan's last lane).
template <typename T, typename Op>
__device__ __forceinline__ T wave_reduce(T x, T none, Op op)
{
    return lane_value(wave_scan(x, none, op), kWave - 1);
}

// Inclusive prefix sum across the wave.
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x)
{
    return wave_scan(x, 0u, [](uint32_t a, uint32_t b) { return a + b; });
}

__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t x)
{
    return wave_reduce(x, (uint64_t)0, [](uint64_t a, uint64_t b) { return a + b; });
}

__device__ __forceinline__ double wave_sum_f64(double x)
{
    return wave_reduce(x, 0.0, [](double a, double b) { return a + b; });
}

__device__ __forceinline__ uint32_t wave_min_u32(uint32_t x)
{
    return wave_reduce(x, ~0u, [](uint32_t a, uint32_t b) { return min(a, b); });
}

__device__ __forceinline__ uint32_t wave_max_u32(uint32_t x)
{
    return wave_reduce(x, 0u, [](uint32_t a, uint32_t b) { return max(a, b); });
}

// Append `v` to q (counter *cnt) for every lane with `pred`, one atomic per wave.
// Must be reached by the whole wave (convergent), with per-lane predicates.
__device__ __forceinline__ void wave_append(bool pred, uint32_t v, uint32_t *q, uint32_t *cnt)
{
    uint64_t m = ballot(pred);
    if (!m) return;
    int leader = first_lane(m);
    uint32_t base = 0;
    if (lane() == leader) base = atomicAdd(cnt, (uint32_t)__popcll(m));
    base = lane_value(base, leader);
    if (pred) q[base + rank_in(m)] = v;
}

// ---------------------------------------------------------------- grid barrier
// A grid barrier for persistent kernels whose blocks are all resident.
//
// Blocks are grouped by the XCD they physically run on (hardware register
// XCC_ID; each XCD has its own L2). Data produced before the barrier reaches
// the writer's L2 when the block's waves pass __syncthreads (vector L1 is
// write-through); the last block to arrive on an XCD writes that L2 back once
// (agent-scope release) and signals the top counter, so the barrier costs one
// L2 write-back per XCD instead of one per block. The last XCD flips the
// generation word, which every block polls (system scope, so no cache can
// answer) before its agent-scope acquire. Relaying the flip through a per-XCD
// flag set by the XCD's leader measured slower on MI355X (one more store/poll
// hop on the critical path).
//
// Counters come in two sets used by alternate barriers (generation parity).
// A set's counters are zeroed by the blocks that finished with them -- the
// XCD leader after its top arrival, the last XCD after the flip -- and those
// stores drain before the same blocks arrive at the next barrier, so they
// land before the set is used again two barriers on. No store has to
// complete between the last arrival and the flip.
//
// How many blocks each XCD holds is counted on every launch: each block
// registers on its XCD when it starts (bar_begin), and before its first
// barrier a block waits until the whole grid has registered and reads the
// per-XCD counts (the census). Registration counters come in two sets chosen
// by the launch's parity (GridBarrier::rset); block 0 zeroes the other set,
// which only the previous launch on these words used, when it starts. So no
// launch depends on how blocks were dispatched in an earlier one.
constexpr int kBarLine = 32;      // uint32 per 128-byte line
constexpr int kMaxXcd = 16;       // XCC_ID is 4 bits wide
constexpr int kBarWords = kBarLine * (21 + 4 * kMaxXcd);

// Word offsets inside the barrier area.
constexpr int kBarGen = 0;
constexpr int kBarStamp = 2;  // 64-bit: wall clock when a stamped barrier completed
__host__ __device__ constexpr int bar_top(int set) { return kBarLine * (1 + set); }
__host__ __device__ constexpr int bar_arrive(int set, int x) { return kBarLine * (3 + set * kMaxXcd + x); }
__host__ __device__ constexpr int bar_count(int x) { return kBarLine * (3 + 2 * kMaxXcd) + x; }
// residency probe: blocks registered / blocks whose wait for the others expired
constexpr int kBarProbeTotal = kBarLine * (3 + 2 * kMaxXcd) + kMaxXcd;
constexpr int kBarProbeFail = kBarProbeTotal + 1;
// per-launch registration: blocks on XCD x, per parity set
__host__ __device__ constexpr int bar_reg(int set, int x) { return kBarLine * (4 + 2 * kMaxXcd + set * kMaxXcd + x); }
// team rounds: the members' words, per launch parity and round parity, and the
// notes a team leaves for the rest of the grid when its phase ends
constexpr uint32_t kTeamMax = 32;
__host__ __device__ constexpr int bar_slots(int set) { return kBarLine * (4 + 4 * kMaxXcd + 8 * set); }
constexpr int kBarNote = kBarLine * (20 + 4 * kMaxXcd);
static_assert(bar_slots(1) - bar_slots(0) == 2 * 2 * kTeamMax * 2, "team words layout");
static_assert(kBarNote + kBarLine <= kBarWords, "barrier layout");

struct GridBarrier {
    uint32_t *words;          // kBarWords, zero-initialised counters
    uint32_t spin_limit;      // max polls before giving up (sets *abort)
    uint32_t rset;            // registration set of this launch (launch parity)
    uint64_t *clock = nullptr;  // optional [1 + blocks]: wall clock at block 0's start, at each block's end
};

// Barrier state kept by thread 0 of each block.
struct BarState {
    uint32_t gen;   // generation the next barrier completes from
    uint32_t cnt;   // blocks of the grid on this block's XCD (0 before the census)
    uint32_t nxcd;  // XCDs holding at least one block of the grid
    uint32_t rank;  // this block's arrival order among its XCD's blocks
    uint32_t first; // lowest XCD holding blocks of the grid (the team's)
    uint32_t ok;    // what grid_signal found
};

__device__ __forceinline__ uint32_t xcc_id() { return __builtin_amdgcn_s_getreg((3 << 11) | 20) & 15; }

__device__ __forceinline__ uint32_t atomic_load_relaxed(const uint32_t *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void atomic_store_relaxed(uint32_t *p, uint32_t v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ uint32_t atomic_add_relaxed(uint32_t *p, uint32_t v)
{
    return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Loads and stores of flags that another block changes while this one waits.
// An agent-scope atomic load (sc1 only) can keep hitting a cached copy across
// polls on gfx950 -- observed as barrier waits that never saw a release -- so
// polling uses system scope (sc0 sc1), which no cache level may satisfy.
__device__ __forceinline__ uint32_t poll_load(const uint32_t *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ void flag_store(uint32_t *p, uint32_t v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Bounded wait until *p != v (want_ne) or *p == v (!want_ne). kLong: the wait
// may last many rounds (a team phase), so the polls are spaced out.
template <bool kLong = false>
__device__ __forceinline__ bool spin_wait(const uint32_t *p, uint32_t v, bool want_ne, uint32_t limit,
                                          uint32_t *abort)
{
    uint32_t polls = 0;
    for (;;) {
        const uint32_t x = poll_load(p);
        if (want_ne ? x != v : x == v) return true;
        if ((++polls & 63) == 0 && poll_load(abort)) return false;
        if (polls > limit) {
            flag_store(abort, 1u);
            return false;
        }
        __builtin_amdgcn_s_sleep(kLong ? 8 : 1);
    }
}

// End of a persistent kernel that the engine times: the run took from block
// 0's start to the end of the last block's last wave, its stores done. Reached
// by every wave of the block. Two event records around the kernel took
// 7 us of every call (RMAT-12 BFS 35.5 us with them, 28.3 without), these
// stores cost none that could be measured.
__device__ __forceinline__ void bar_end(const GridBarrier &gb)
{
    if (!gb.clock) return;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) gb.clock[1 + blockIdx.x] = (uint64_t)wall_clock64();
}

// Start of a persistent kernel (thread 0's copy is the one used): read the
// generation, register this block on its XCD, and let block 0 zero the
// registration set (and, with kTeam, the team words) of the other parity for
// the next launch.
template <bool kTeam = false>
__device__ __forceinline__ BarState bar_begin(const GridBarrier &gb, uint32_t xcc)
{
    BarState s{0u, 0u, 0u, 0u, 0u, 0u};
    if (kTeam && blockIdx.x == 0 && threadIdx.x < 4 * kTeamMax)
        ((uint64_t *)(gb.words + bar_slots((int)(gb.rset & 1u) ^ 1)))[threadIdx.x] = 0;
    if (threadIdx.x == 0) {
        if (gb.clock && blockIdx.x == 0) gb.clock[0] = (uint64_t)wall_clock64();
        uint32_t *w = gb.words;
        const int set = (int)(gb.rset & 1u);
        s.gen = poll_load(w + kBarGen);
        s.rank = atomic_add_relaxed(w + bar_reg(set, (int)xcc), 1u);
        if (blockIdx.x == 0) {
            for (int x = 0; x < kMaxXcd; x++) flag_store(w + bar_reg(set ^ 1, x), 0u);
        }
    }
    return s;
}

// The census (thread 0): bounded wait until every block of the grid has
// registered, then the blocks per XCD (all[x], when given) and this block's
// share. Every block adds one to one XCD's counter, so the counts are final
// once they sum to the grid. (A total of its own beside them is one word that
// every block adds to, 11 ns each: with it, a launch of 256 blocks took 3 us longer.)
__device__ inline bool bar_census(const GridBarrier &gb, uint32_t xcc, BarState &s, uint32_t *abort,
                                  uint32_t *all = nullptr)
{
    const uint32_t *w = gb.words;
    const int set = (int)(gb.rset & 1u);
    uint32_t polls = 0;
    for (;;) {
        uint32_t c[kMaxXcd];
#pragma unroll
        for (int x = 0; x < kMaxXcd; x++) c[x] = poll_load(w + bar_reg(set, x));
        uint32_t sum = 0, nx = 0;
#pragma unroll
        for (int x = 0; x < kMaxXcd; x++) {
            sum += c[x];
            nx += c[x] != 0u;
        }
        if (sum == gridDim.x) {
            s.cnt = c[xcc];
            s.nxcd = nx;
            s.first = 0;
#pragma unroll
            for (int x = kMaxXcd - 1; x >= 0; x--)
                if (c[x]) s.first = (uint32_t)x;
            if (all)
                for (int x = 0; x < kMaxXcd; x++) all[x] = c[x];
            return true;
        }
        if ((++polls & 63) == 0 && poll_load(abort)) return false;
        if (polls > gb.spin_limit) {
            flag_store(abort, 1u);
            return false;
        }
        __builtin_amdgcn_s_sleep(1);
    }
}

// Residency probe, run by a persistent kernel launched with its real grid and
// resources before first use: every block counts itself on its XCD and then
// waits (bounded) until all blocks of the grid have done so. A block whose
// wait expires records a failure: the grid is then larger than what can be
// co-resident and the host shrinks it. Every block exits either way. All of
// a block's waves stay alive until thread 0 is done (the closing
// __syncthreads), so a probe block occupies exactly the wave slots, registers
// and LDS of a working block.
__device__ inline void residency_probe(uint32_t *words, uint32_t limit)
{
    if (threadIdx.x == 0) {
        atomicAdd(&words[bar_count(xcc_id())], 1u);
        atomicAdd(&words[kBarProbeTotal], 1u);
        uint32_t polls = 0;
        while (poll_load(&words[kBarProbeTotal]) < gridDim.x) {
            if (++polls > limit) {
                atomicAdd(&words[kBarProbeFail], 1u);
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
    }
    __syncthreads();
}

// Arrival of this block at the grid barrier (thread 0, after the block's stores
// have drained and the census is taken); returns the generation it ends.
// `closed`: set when it was the last block's.
// kStamp: the block that completes the barrier also records the wall clock
// (barrier_stamp), so every block can time the grid's rounds identically.
template <bool kStamp = false>
__device__ __forceinline__ uint32_t grid_arrive(const GridBarrier &gb, uint32_t xcc, BarState &st,
                                                uint32_t *closed = nullptr)
{
    uint32_t *w = gb.words;
    const uint32_t gen0 = st.gen;
    st.gen = gen0 + 1;
    const int set = (int)(gen0 & 1u);
    uint32_t *arr = w + bar_arrive(set, (int)xcc);
    uint32_t *top = w + bar_top(set);
    const uint32_t a = atomic_add_relaxed(arr, 1u);
    if (a == st.cnt - 1) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        const uint32_t t = atomic_add_relaxed(top, 1u);
        flag_store(arr, 0u);  // this set is used again two barriers on
        if (t == st.nxcd - 1) {
            if (kStamp) {
                // the stamp must be visible before the flip that publishes it
                __hip_atomic_store((uint64_t *)(w + kBarStamp), (uint64_t)wall_clock64(), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_SYSTEM);
                __builtin_amdgcn_s_waitcnt(0);
            }
            flag_store(w + kBarGen, gen0 + 1);
            flag_store(top, 0u);
            if (closed) *closed = 1u;
        }
    }
    return gen0;
}

// The first half of grid_sync: what this block stored before it is there for
// every block that has returned from the grid_wait that follows. Work between
// the two hides the wait for the other blocks.
template <bool kStamp = false>
__device__ __forceinline__ void grid_signal(const GridBarrier &gb, uint32_t xcc, BarState &st, uint32_t *abort)
{
    // __syncthreads() alone only waits for LDS traffic: every wave must first
    // drain its outstanding global stores/atomics (vmcnt) so they are in the
    // XCD's L2 before the leader writes that L2 back.
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) {
        st.ok = st.cnt != 0u || bar_census(gb, xcc, st, abort);
        if (st.ok) grid_arrive<kStamp>(gb, xcc, st);
    }
}

// Returns false if the wait timed out or another block aborted; the caller
// must then leave its loop.
__device__ __forceinline__ bool grid_wait(const GridBarrier &gb, BarState &st, uint32_t *abort)
{
    __shared__ uint32_t s_ok;
    if (threadIdx.x == 0) {
        // every block polls the generation word itself (a relay through a
        // per-XCD flag costs one more store/poll hop on the critical path)
        uint32_t ok = st.ok;
        if (ok) ok = spin_wait(gb.words + kBarGen, st.gen - 1, true, gb.spin_limit, abort);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        __builtin_amdgcn_s_waitcnt(0);
        s_ok = ok;
    }
    __syncthreads();
    return s_ok != 0;
}

// `st` is this block's state from bar_begin (only thread 0's copy is used):
// the first barrier of a launch takes the census, and each barrier advances
// the generation.
template <bool kStamp = false>
__device__ __forceinline__ bool grid_sync(const GridBarrier &gb, uint32_t xcc, BarState &st, uint32_t *abort)
{
    grid_signal<kStamp>(gb, xcc, st, abort);
    return grid_wait(gb, st, abort);
}

// Wall clock recorded by the last stamped barrier (read after it).
__device__ __forceinline__ uint64_t barrier_stamp(const GridBarrier &gb)
{
    return __hip_atomic_load((const uint64_t *)(gb.words + kBarStamp), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------- team rounds
// A round with little work costs its fixed parts. A grid barrier takes 3.6 us
// on MI355X, ~1.9 of them every block's agent-scope acquire, which also leaves
// each XCD's L2 cold: every dependent load of the next round then goes to
// memory (0.4-0.8 us against ~0.12 from L2). Such rounds run on the blocks of one
// XCD, the team, while the others wait at the next grid barrier. A team's
// traffic meets in that XCD's L2, so its barrier needs neither write-back nor
// invalidation, and the graph stays in L2 from round to round: 0.97 us a
// barrier for 32 blocks (1.4 us with a store before and a read after it).
//
// What replaces the invalidation: in a team round, words that other blocks
// change are read with agent-scope loads (load_team), which pass by the CU's
// L1 and are served by the L2. Stores are in L2 once vmcnt has drained, and
// atomics execute there. 98 M words changed by atomicMin, atomicOr and plain
// stores and read by other CUs after the barrier: plain loads found ~200 of
// them stale (L1), agent-scope loads none.
template <typename T>
__device__ __forceinline__ T load_team(const T *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A member's word: what its block found in the round, and the round's tag.
constexpr int kTeamCountShift = 32, kTeamFlagShift = 51, kTeamTagShift = 52;
constexpr uint64_t kTeamCountMask = (1ull << (kTeamFlagShift - kTeamCountShift)) - 1;

// LDS of a team round.
struct TeamLds {
    unsigned long long slot[2 * kTeamMax];  // every member's words of the last round
    unsigned long long acc;                 // this round: sum in bits 0..31, count above
    uint32_t flag, mn, ok;

    // by thread 0, before the launch's first block barrier
    __device__ __forceinline__ void reset()
    {
        acc = 0;
        flag = 0;
        mn = ~0u;
    }
};

// First half of a team round's end: publishes this block's sums (acc, flag
// and, with kMin, the minimum mn), its stores before. Two sets of words in
// turn, as a member may still be polling the last round's.
template <bool kMin = false>
__device__ __forceinline__ void team_arrive(const GridBarrier &gb, const TeamLds &t, uint32_t rank, uint32_t &tag)
{
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    tag++;
    const uint32_t ln = threadIdx.x;
    if (ln == 0 || (kMin && ln == kTeamMax)) {
        uint64_t *slots = (uint64_t *)(gb.words + bar_slots((int)(gb.rset & 1u))) + (tag & 1u) * 2 * kTeamMax;
        const uint64_t mine = ln ? (uint64_t)t.mn : t.acc | (uint64_t)(t.flag != 0u) << kTeamFlagShift;
        __hip_atomic_store(slots + ln + rank, mine | (uint64_t)(tag & 0xFFFu) << kTeamTagShift, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
    }
}

// Second half: waits for every member's words, left in t.slot (the minima from
// kTeamMax on), and resets this block's sums. The words double as the
// barrier: one store and one poll of a few cache lines, no atomics and no
// separate read of the counters. False when the wait expired or a block aborted.
template <bool kMin = false>
__device__ __forceinline__ bool team_wait(const GridBarrier &gb, TeamLds &t, uint32_t members, uint32_t tag,
                                          uint32_t *abort)
{
    if (threadIdx.x < kWave) {
        const uint64_t *slots = (const uint64_t *)(gb.words + bar_slots((int)(gb.rset & 1u))) + (tag & 1u) * 2 * kTeamMax;
        const uint64_t want = tag & 0xFFFu;
        const uint32_t ln = threadIdx.x;
        const bool read = ln % kTeamMax < members && (kMin || ln < kTeamMax);
        uint32_t polls = 0, ok = 1u;
        uint64_t v;
        for (;;) {
            v = read ? load_team(slots + ln) : want << kTeamTagShift;
            if (!ballot(v >> kTeamTagShift != want)) break;
            if ((++polls & 255) == 0 && poll_load(abort)) {
                ok = 0u;
                break;
            }
            if (polls > gb.spin_limit) {
                flag_store(abort, 1u);
                ok = 0u;
                break;
            }
        }
        t.slot[ln] = read ? v : ln < kTeamMax ? 0ull : ~0ull;
        if (ln == 0) {
            t.reset();
            t.ok = ok;
        }
    }
    __syncthreads();
    return t.ok != 0;
}

// Ends a team round.
template <bool kMin = false>
__device__ __forceinline__ bool team_exchange(const GridBarrier &gb, TeamLds &t, uint32_t members, uint32_t rank,
                                              uint32_t &tag, uint32_t *abort)
{
    team_arrive<kMin>(gb, t, rank, tag);
    return team_wait<kMin>(gb, t, members, tag, abort);
}

// A member's place in a team phase, and the frontier as segments of a queue,
// one per block that found its vertices (lane k holds the entries up to the
// end of segment k).
struct TeamFront {
    uint32_t members, rank, tag;
    uint32_t gwave, nwaves;
    uint32_t incl, total;  // segment ends (by lane), entries in all
    uint32_t seg;          // entries per segment
    const uint32_t *qin;
    uint32_t *qout;        // this block's segment of the next queue
};

// What an exchange left: segment ends, entries in all; returned: this lane's word.
__device__ __forceinline__ uint64_t team_segments(TeamFront &T, const TeamLds &t)
{
    const uint64_t w = (uint32_t)lane() < kTeamMax ? t.slot[lane()] : 0ull;
    T.incl = wave_incl_scan((uint32_t)((w >> kTeamCountShift) & kTeamCountMask));
    T.total = lane_value(T.incl, kWave - 1);
    return w;
}

// Queue entry i of each lane (i >= T.total: 0), i0 the wave's lowest. The
// segment is found for i0 by one ballot and stepped on from there.
// Wave-convergent.
__device__ __forceinline__ uint32_t team_entry(const TeamFront &T, uint32_t i0, uint32_t i)
{
    int k = __popcll(ballot(T.incl <= i0));
    for (;;) {
        const uint32_t stop = shfl(T.incl, k);
        const bool past = i < T.total && i >= stop;
        if (!ballot(past)) break;
        k += past;
    }
    const uint32_t before = shfl(T.incl, k > 0 ? k - 1 : 0);
    return i < T.total ? load_team(T.qin + (size_t)k * T.seg + (i - (k > 0 ? before : 0u))) : 0u;
}

// Lanes per item (a power of two from 4 to 64, as its logarithm) that give
// `items` the team's lanes once over.
__device__ __forceinline__ uint32_t team_width(const TeamFront &T, uint32_t items)
{
    uint32_t shift = 6;
    while (shift > 2 && ((uint64_t)items << shift) > (uint64_t)T.nwaves * kWave) shift--;
    return shift;
}

// Adds v (out-degree dv) to this block's segment of the next queue.
__device__ __forceinline__ void team_append(const TeamFront &T, TeamLds &t, uint32_t v, uint32_t dv)
{
    const unsigned long long old = atomicAdd(&t.acc, (1ull << kTeamCountShift) | dv);
    T.qout[(uint32_t)(old >> kTeamCountShift)] = v;
}

// This member's share of the frontier bitmap `bits` into its segment `q`; an
// exchange follows.
__device__ __forceinline__ void team_gather(TeamLds &t, const uint64_t *bits, uint32_t words, uint32_t *q, uint32_t tid,
                                            uint32_t nthreads)
{
    for (uint32_t w = tid; w < words; w += nthreads) {
        uint64_t x = load_team(bits + w);
        if (!x) continue;
        const unsigned long long old = atomicAdd(&t.acc, (unsigned long long)__popcll(x) << kTeamCountShift);
        uint32_t at = (uint32_t)(old >> kTeamCountShift);
        for (; x; x &= x - 1) q[at++] = w * 64 + (uint32_t)first_lane(x);
    }
}

}  // namespace sg
