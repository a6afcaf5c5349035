// Device side of the hybrid (direction-switching) BFS: one query runs as a
// persistent grid (a whole launch, or the blocks of one XCD).
//
// Reference path (samples/hybrid_bfs/hybrid_bfs.cu:173-243 driving
// Engine::Start, include/framework/framework.cuh:315-375): each round the host
// converts the frontier between a queue and a bitmap, counts it, sums its
// out-degree, launches AsyncPushDD (queue, CSR out-edges,
// include/framework/variants/async_push_dd.cuh:79-147) or AsyncPullDD (bitmap,
// CSC in-edges with early exit, async_pull_dd.cuh:26-70), and asks
// PolicyDecisionMaker::GetNextPolicy (include/framework/hybrid_policy.h:237-291)
// for the next direction -- at least six blocking host round trips per round.
//
// Here the whole traversal is one launch. Every block evaluates the same
// alpha/beta rule on device from counters read after a grid barrier, so no
// round needs the host. Per vertex, a push round writes the level and two
// bits:
//   * discovery: an edge whose head shows an unset bit in the visited filter
//     claims that bit (one returning atomicOr per run of a wave's candidates
//     in one word, none per edge); the claimer stores level L+1 and queues the
//     vertex. The reference's default non-atomic BFS min
//     (hybrid_bfs.cu:128-134, hybrid_bfs/main.cpp:37) lets racing writers
//     queue a vertex several times; claiming keeps the queue exact, which
//     matters on high-diameter graphs where duplicates compound round after
//     round. Candidates also set the next frontier's bitmap, so visited and
//     frontier tests read 512 KiB of L2-resident bits, never the level array;
//   * the next queue is staged in LDS per block and published with one
//     atomic per block per round (same-address atomics serialise on MI355X);
//   * vertices with out-degree > kHugeDegree are expanded through the graph's
//     static chunk list, filtered by membership, so hub adjacencies spread
//     over every wave without building any list at run time.
// A pull round sweeps 64-vertex words (dealt round-robin over the waves,
// kPullGroup words at a time): every unvisited lane tests its first
// in-neighbour from the graph's head array, then the group's words walk their
// remaining in-edge lists in lock step, 64 edges per word per step with all
// of the group's loads in flight together, re-planning after each step so a
// vertex stops at its first parent (the reference's early break,
// pull_functor.h:138-188). Pull rounds write whole words of the next frontier
// bitmap and of a visited filter, so they need no atomics.
//
// Rounds with little work, and whole queries on small graphs, run on the blocks
// of one XCD, the team, with a barrier inside its L2 (bfs_team_phase,
// bfs_whole; team_exchange in sg_device.hpp).
#pragma once

#include "frontier.hpp"

using namespace sg;

// Words of 64 vertices a wave works on at once in a pull round.
#ifndef SG_PULL_GROUP
#define SG_PULL_GROUP 2
#endif
// Minimum waves per SIMD the compiler must allow for k_bfs (0: no bound);
// 8 caps registers at 64 so two 1024-thread blocks fit on a CU.
#ifndef SG_BFS_WAVES
#define SG_BFS_WAVES 0
#endif

namespace {
namespace bfsk {

constexpr int kPullGroup = SG_PULL_GROUP;

struct BfsArgs {
    DevGraph g;
    // levels in the caller's vertex order: device vertex v's level goes to
    // level[perm[v]] (perm null: the orders agree). Nothing reads it during
    // the traversal (visited tests use the filter), so a degree-ordered graph
    // needs no device-order copy and no gather at the end.
    int32_t *level;
    const uint32_t *perm;
    uint64_t *vis;    // W words: visited filter (set bit => visited or in-degree 0)
    uint64_t *vis_idle;  // the other filter, reset here for the next query
    uint64_t *fbit;   // 3 * W words: frontier L's bitmap in slot L % 3
    uint32_t *queue;  // 3 * qcap entries
    uint32_t qcap;
    FrontierCtr *ctr; // 3 slots
    GridBarrier bar;
    uint32_t *abort;
    DevStats *stats;
    DevTrace *trace;
    uint32_t source;     // device vertex id
    uint32_t source_id;  // the caller's id of the same vertex
    int32_t force;    // -1 auto, 0 push, 1 pull
    double alpha, beta;
    uint32_t total_workload0;
    uint32_t max_rounds;
    uint32_t probe;   // launch is a residency probe of the grid
    uint32_t full_init;  // bitmaps and counters not known to be clean
    // LoadBalancing::NONE (one lane per vertex, its edges in order, no hub
    // chunks) for push / pull rounds; otherwise the balanced schedulers
    uint32_t lb_push_none, lb_pull_none;
    uint32_t team;        // rounds with little work may run on one XCD's blocks:
                          // 1 (skewed graphs) after the first pull round, 2 from the start
    uint32_t team_start;  // (2) see team_start()
};

// Hub chunks whose heads a block stages in LDS at a time (with 64-edge
// chunks: 4096 heads, 16 KiB), and the mark of a staged slot past a chunk's end.
constexpr uint32_t kStageChunks = 64;
// Member chunks a block lists before staging them (16 KiB of LDS).
constexpr uint32_t kHubList = 2048;
constexpr uint32_t kNoHead = 0xFFFFFFFFu;
static_assert(kHugeChunk <= kWave, "a staged hub chunk is expanded by one wave in one step");

// Largest source out-degree whose expansion (round 0) block 0 does alone.
constexpr uint32_t kLocalRound0 = 4096;

__device__ __forceinline__ uint32_t caller_id(const BfsArgs &a, uint32_t v) { return a.perm ? a.perm[v] : v; }

struct Round {
    const BfsArgs *a;
    int32_t L;              // level being expanded
    const uint64_t *fcur;   // frontier L as a bitmap
    uint64_t *fnext;        // frontier L+1, built by this round
    Stager S;
    unsigned long long scout, count;  // this lane's share of the next frontier
    bool huge;                        // this lane discovered a vertex above kHugeDegree
    bool levels = true;               // write discovered levels now (else the next round does)
    bool even = false;                // bfs_run's kEven
};

__device__ __forceinline__ bool in_frontier(const Round &R, uint32_t u) { return test_bit(R.fcur, u); }

// Push edge -> v for `act` lanes; wave-convergent.
__device__ __forceinline__ void push_visit(Round &R, bool act, uint32_t v)
{
    const BfsArgs &a = *R.a;
    // candidates: not visited as far as this lane can see (bits set by other
    // waves in this round may not be visible yet). Claiming the bit in the
    // visited filter picks one discoverer; every candidate was unvisited
    // before this round, so all of them belong in the next frontier's bitmap.
    // Visited tests here and membership tests in a pull round read 512 KiB
    // of L2-resident bits instead of the level array, with one atomic per
    // run of a wave's candidates in one word, none per edge.
    const bool cand = act && !test_bit(a.vis, v);
    const bool found = R.even ? wave_claim_bits<true>(a.vis, cand, v, R.fnext) : wave_claim_bits(a.vis, cand, v, R.fnext);
    if (found) {
        if (R.levels) a.level[caller_id(a, v)] = R.L + 1;
        const uint32_t dv = a.g.row[v + 1] - a.g.row[v];
        R.scout += dv;
        R.count++;
        R.huge |= dv > kHugeDegree;
    }
    stage(R.S, found, v);
}

// Expand the out-edges of up to 64 vertices (one per lane) with wave-level
// prefix-sum scheduling: 64 consecutive edges of the concatenated adjacency
// per step, so CSR reads are coalesced and lanes stay busy. Vertices above
// kHugeDegree are left to the chunk list.
__device__ __forceinline__ void push_expand(Round &R, bool valid, uint32_t u)
{
    const DevGraph &g = R.a->g;
    uint32_t b = 0, d = 0;
    if (valid) {
        b = g.row[u];
        d = g.row[u + 1] - b;
        if (d > kHugeDegree) d = 0;
    }
    const uint32_t incl = wave_incl_scan(d);
    const uint32_t total = lane_value(incl, kWave - 1);
    const uint32_t off = b - (incl - d);
    const int ln = lane();
    for (uint32_t jb = 0; jb < total; jb += kWave) {
        const uint32_t j = jb + ln;
        const bool act = j < total;
        const int k = owner_lane(incl, j);
        const uint32_t e = shfl(off, k) + j;
        push_visit(R, act, act ? g.col[e] : 0u);
    }
}

// LoadBalancing::NONE push: each lane walks its own vertex's out-edges in
// CSR order, hubs included (the reference's thread-per-vertex relax,
// async_push_dd.cuh:24-78); the wave steps through the longest list.
__device__ __forceinline__ void push_expand_serial(Round &R, bool valid, uint32_t u)
{
    const DevGraph &g = R.a->g;
    uint32_t b = 0, d = 0;
    if (valid) {
        b = g.row[u];
        d = g.row[u + 1] - b;
    }
    uint32_t dmax = d;
    dmax = wave_max_u32(dmax);
    for (uint32_t j = 0; j < dmax; j++) {
        const bool act = j < d;
        push_visit(R, act, act ? g.col[b + j] : 0u);
    }
}

// LoadBalancing::NONE pull for the word `w` (visited word vw): each
// unvisited lane walks its own in-edges in CSC order and stops at its first
// parent in the frontier (async_pull_dd.cuh:26-70).
__device__ __forceinline__ void pull_word_serial(Round &R, uint32_t w, uint64_t vw)
{
    const BfsArgs &a = *R.a;
    const DevGraph &g = a.g;
    const int ln = lane();
    const uint32_t v = w * 64 + ln;
    const uint64_t visited = ballot(v >= g.n) | vw;
    const bool want = !((visited >> ln) & 1);
    uint32_t b = want ? g.cstart[v] : 0u, e = want ? g.cstart[v + 1] : 0u;
    bool found = false;
    while (ballot(b < e && !found)) {
        if (b < e && !found) {
            found = in_frontier(R, g.csrc[b]);
            b++;
        }
    }
    const uint64_t fm = ballot(found);
    if (ln == 0) {
        a.vis[w] = visited | fm;
        R.fnext[w] = fm;
        R.count += __popcll(fm);
    }
    if (found) {
        a.level[caller_id(a, v)] = R.L + 1;
        const uint32_t dv = g.row[v + 1] - g.row[v];
        R.scout += dv;
        R.huge |= dv > kHugeDegree;
    }
}

// Bottom-up step for the 64 vertices of each of ng (<= G) words wg[i] (vwg[i]:
// visited filter word). Every load of a stage is issued for all G words
// before any is used, so the words' dependent chains overlap.
template <int G>
__device__ __forceinline__ void pull_group(Round &R, const uint32_t (&wg)[G], const uint64_t (&vwg)[G], int ng)
{
    const BfsArgs &a = *R.a;
    const DevGraph &g = a.g;
    const int ln = lane();
    uint32_t v[G], b[G], e[G], u[G];
    uint64_t visited[G];
    bool found[G];
#pragma unroll
    for (int i = 0; i < G; i++) v[i] = wg[i] * 64 + ln;
    bool want[G];
    uint32_t dv[G];
    // One step issues, for every unvisited lane, the first in-neighbour (from
    // the head array, coalesced across the word), the in-edge range and the
    // out-degree, so the parent test, the walk and the frontier statistics
    // wait on a single round of loads.
#pragma unroll
    for (int i = 0; i < G; i++) {
        // the filter holds every discovery (pull rounds write whole words,
        // push rounds set bits), the inert vertices and the source
        visited[i] = i < ng ? (ballot(v[i] >= g.n) | vwg[i]) : ~0ull;
        want[i] = !((visited[i] >> ln) & 1);
        u[i] = want[i] ? g.chead[v[i]] : 0xFFFFFFFFu;
        b[i] = want[i] ? g.cstart[v[i]] : 0u;
        e[i] = want[i] ? g.cstart[v[i] + 1] : 0u;
        dv[i] = want[i] ? g.row[v[i] + 1] - g.row[v[i]] : 0u;
    }
#pragma unroll
    for (int i = 0; i < G; i++) {
        found[i] = u[i] != 0xFFFFFFFFu && in_frontier(R, u[i]);
        // lanes still looking walk their in-edges past the head
        if (found[i] || u[i] == 0xFFFFFFFFu) b[i] = e[i];
        else b[i]++;
    }
    // Walk the remaining in-edge lists of every word of the group in lock
    // step: each iteration plans one 64-edge step per word (the concatenated
    // lists of its still-searching lanes), then issues all of the group's
    // loads before any test, so one memory latency covers G steps. A lane
    // stops at its first parent (re-planned every step).
    for (;;) {
        uint32_t idx[G], incl[G], excl[G];
        bool valid[G];
        bool any = false;
#pragma unroll
        for (int i = 0; i < G; i++) {
            const uint32_t r = found[i] ? 0u : e[i] - b[i];
            incl[i] = wave_incl_scan(r);
            excl[i] = incl[i] - r;
            const uint32_t total = lane_value(incl[i], kWave - 1);
            any |= total != 0;
            valid[i] = (uint32_t)ln < total;
            const int k = owner_lane(incl[i], valid[i] ? (uint32_t)ln : 0u);
            idx[i] = shfl(b[i], k) + ((uint32_t)ln - shfl(excl[i], k));
        }
        if (!any) break;
        uint32_t src[G];
#pragma unroll
        for (int i = 0; i < G; i++) src[i] = valid[i] ? g.csrc[idx[i]] : 0u;
#pragma unroll
        for (int i = 0; i < G; i++) {
            const uint64_t H = ballot(valid[i] && in_frontier(R, src[i]));
            const uint32_t lo = min(excl[i], 64u), hi = min(incl[i], 64u);
            if (hi > lo) {
                const uint32_t c = hi - lo;
                const uint64_t msk = (c == 64 ? ~0ull : ((1ull << c) - 1)) << lo;
                if (H & msk) found[i] = true;
                b[i] += c;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < G; i++) {
        if (i >= ng) break;
        const uint64_t fm = ballot(found[i]);
        if (ln == 0) {
            a.vis[wg[i]] = visited[i] | fm;
            R.fnext[wg[i]] = fm;
            R.count += __popcll(fm);
        }
        if (found[i]) {
            a.level[caller_id(a, v[i])] = R.L + 1;
            R.scout += dv[i];
            R.huge |= dv[i] > kHugeDegree;
        }
    }
}

// ------------------------------------------------------------ team rounds
// On a graph that the team runs whole, every member keeps the visited filter
// and the round's frontier in LDS (2 x 2 KiB; the frontier's vertices are counted
// off its bitmap, so there is no queue), and the rounds meet only in the
// next frontier's bitmap: atomics on the few cache lines such bitmaps fill
// serialise (6-15 ns each on one line), so a bit set in a member's own copy
// is claimed there first.

// Edges of a narrow push round at most.
#ifndef SG_TEAM_PUSH_EDGES
#define SG_TEAM_PUSH_EDGES 16384
#endif
constexpr uint32_t kTeamPushEdges = SG_TEAM_PUSH_EDGES;

// Whether round L, of a grid round's frontier, starts a team phase; evaluated
// alike by every block. Only narrow push rounds do: on the 2048 x 2048 grid
// (2668 rounds of at most 10.6 K edges) they take 4.4-6.1 us on the team and
// 10.2-11.4 on the whole grid, 33.6 -> 16.3 ms a query; with the limit at 8 K
// edges it takes 17.3 ms, at 4 K 24.5, and no measured graph had a round between
// 16 K and 32 K that told them apart.
// On a skewed graph only once its peak is past: before it a
// narrow frontier's next one is seldom narrow, and ending a phase costs a
// barrier and a frontier read back from its bitmap; and only when nothing
// follows the traversal (kLeave): its last one to three rounds do not earn
// the barrier back (the BFS of a BC query on 32 001 vertices: 230 us without, 238 with).
template <bool kLeave, bool kEven>
__device__ __forceinline__ bool bfs_team_fits(const BfsArgs &a, const RoundState &S, const RoundCounts &rc, uint32_t prev)
{
    if (!a.team) return false;
    const uint32_t limit = team_limit(a.qcap, kTeamPushEdges);
    DirectionPolicy p = S.pol;
    const bool stays =
        kEven ? team_stays(a.team_start, rc.count, prev, rc.scout) : a.team == 2 || (kLeave && S.pulls);
    return stays && !rc.has_huge && rc.count <= limit && rc.scout <= limit &&
           !p.next(S.L, rc.count, rc.scout);
}

// What the rounds of a phase share.
struct BfsTeam : TeamFront {
    uint32_t L;
    uint64_t *fnext;
    TeamBits *front;         // whole-graph phases: frontier L and the visited
    uint64_t *s_vis;         // filter in LDS
};

// A vertex found for level L+1: its level, its share of the sums and its place
// in the next queue (a whole-graph phase has none). `dv`: its out-degree.
template <bool kWhole>
__device__ __forceinline__ void team_found(const BfsArgs &a, const BfsTeam &T, TeamLds &t, uint32_t v, uint32_t id,
                                           uint32_t dv)
{
    a.level[id] = (int32_t)T.L + 1;
    if (dv > kHugeDegree) t.flag = 1u;
    if (kWhole) atomicAdd(&t.acc, (1ull << kTeamCountShift) | dv);
    else team_append(T, t, v, dv);
}

// Edge -> v for `act` lanes. One atomicOr claims an unvisited head (heads of a
// narrow round seldom share a word, so runs are not gathered first); the loads
// a discovery needs travel with it.
template <bool kWhole>
__device__ __forceinline__ void team_visit(const BfsArgs &a, const BfsTeam &T, TeamLds &t, bool act, uint32_t v)
{
    if (!act) return;
    const uint32_t w = v >> 6;
    const uint64_t bit = 1ull << (v & 63);
    uint64_t old;
    if constexpr (kWhole) {
        if (T.s_vis[w] & bit) return;
        if (atomicOr((unsigned long long *)&T.s_vis[w], (unsigned long long)bit) & bit) return;
        old = atomicOr((unsigned long long *)&T.fnext[w], (unsigned long long)bit);
    } else {
        if (load_team(a.vis + w) & bit) return;
        old = atomicOr((unsigned long long *)&a.vis[w], (unsigned long long)bit);
    }
    const uint32_t rb = a.g.row[v], re = a.g.row[v + 1];
    const uint32_t id = caller_id(a, v);
    if (!(old & bit)) team_found<kWhole>(a, T, t, v, id, re - rb);
}

// Push: `width` lanes per queue entry (a power of two, 4 to 64, as many as the
// team has for the frontier), each taking every width-th out-edge, so a
// narrow frontier needs no edge scheduling across the wave.
template <bool kWhole>
__device__ __forceinline__ void team_push(const BfsArgs &a, const BfsTeam &T, TeamLds &t, bool hubs)
{
    const DevGraph &g = a.g;
    const int ln = lane();
    if (kWhole && hubs) {
        // out-degrees above kHugeDegree by the chunk list
        for (uint32_t c0 = 0; c0 < g.nhuge; c0 += T.nwaves * kWave) {
            const uint32_t c = c0 + (uint32_t)ln * T.nwaves + T.gwave;
            uint2 dsc = make_uint2(0u, 0u);
            uint32_t end = 0;
            bool mem = false;
            if (c < g.nhuge) {
                dsc = g.huge[c];
                end = g.huge_end[c];
                mem = test_bit(T.front->word, dsc.x);
            }
            uint64_t mm = ballot(mem);
            while (mm) {
                const int k = first_lane(mm);
                mm &= mm - 1;
                const uint32_t beg = lane_value(dsc.y, k), stop = lane_value(end, k);
                for (uint32_t e = beg + (uint32_t)ln; e < stop; e += kWave)
                    team_visit<kWhole>(a, T, t, true, g.col[e]);
            }
        }
    }
    const uint32_t shift = team_width(T, T.total);
    const uint32_t width = 1u << shift, groups = kWave >> shift;
    const uint32_t grp = (uint32_t)ln >> shift, sub = (uint32_t)ln & (width - 1);
    for (uint32_t i0 = T.gwave * groups; i0 < T.total; i0 += T.nwaves * groups) {
        const uint32_t i = i0 + grp;
        uint32_t u = 0, e = 0, end = 0;
        if (!kWhole) u = team_entry(T, i0, i);
        if (i < T.total) {
            if (kWhole) u = team_bits_entry(*T.front, i);
            e = g.row[u];
            end = g.row[u + 1];
            if (end - e > kHugeDegree) end = e;
            e += sub;
        }
        for (; ballot(e < end); e += 2 * width) {
            const bool p = e < end, q = e + width < end;
            const uint32_t v = p ? g.col[e] : 0u, w = q ? g.col[e + width] : 0u;
            team_visit<kWhole>(a, T, t, p, v);
            team_visit<kWhole>(a, T, t, q, w);
        }
    }
}

// Pull (whole-graph phases): an in-hub per wave, 256 of its in-edges in flight,
// then `width` lanes per other unvisited vertex, a wave's vertices adjacent so
// that it sets their next-frontier bits with one atomic. Each stops at a
// first parent.
__device__ __forceinline__ void team_pull(const BfsArgs &a, const BfsTeam &T, TeamLds &t)
{
    const DevGraph &g = a.g;
    const uint32_t n = g.n;
    const int ln = lane();
    constexpr int K = 4;
    for (uint32_t h = T.gwave; h < g.nhubin; h += T.nwaves) {
        const uint2 first = g.hugein[g.hubin[h].x];
        const uint32_t v = first.x, stop = g.cstart[v + 1];
        if (test_bit(T.s_vis, v)) continue;
        for (uint32_t e0 = first.y; e0 < stop; e0 += K * kWave) {
            uint32_t u[K];
#pragma unroll
            for (int k = 0; k < K; k++) {
                const uint32_t e = e0 + (uint32_t)(k * kWave + ln);
                u[k] = e < stop ? g.csrc[e] : 0xFFFFFFFFu;
            }
            bool hit = false;
#pragma unroll
            for (int k = 0; k < K; k++) hit |= u[k] != 0xFFFFFFFFu && test_bit(T.front->word, u[k]);
            if (!ballot(hit)) continue;
            if (ln == 0) {
                atomicOr((unsigned long long *)&T.fnext[v >> 6], 1ull << (v & 63));
                team_found<true>(a, T, t, v, caller_id(a, v), g.row[v + 1] - g.row[v]);
            }
            break;
        }
    }
    const uint32_t shift = team_width(T, n);
    const uint32_t width = 1u << shift, groups = kWave >> shift;
    const uint32_t grp = (uint32_t)ln >> shift, sub = (uint32_t)ln & (width - 1);
    const uint64_t gmask = (shift == 6 ? ~0ull : (1ull << width) - 1) << (grp << shift);
    for (uint32_t v0 = T.gwave * groups; v0 < n; v0 += T.nwaves * groups) {
        const uint32_t v = v0 + grp;
        const bool want = v < n && !test_bit(T.s_vis, v);
        if (!ballot(want)) continue;
        uint32_t e = 0, end = 0, dv = 0, id = 0;
        if (want) {
            e = g.cstart[v];
            end = g.cstart[v + 1];
            if (end - e > kPullHubDegree) end = e;
            e += sub;
            dv = g.row[v + 1] - g.row[v];
            id = caller_id(a, v);
        }
        bool found = false;
        while (ballot(e < end)) {
            uint32_t u[K];
#pragma unroll
            for (int k = 0; k < K; k++) u[k] = e + k * width < end ? g.csrc[e + k * width] : 0xFFFFFFFFu;
            bool hit = false;
#pragma unroll
            for (int k = 0; k < K; k++) hit |= u[k] != 0xFFFFFFFFu && test_bit(T.front->word, u[k]);
            found |= (ballot(hit) & gmask) != 0;
            e = found ? end : e + K * width;
        }
        found = found && sub == 0;
        if (!ballot(found)) continue;
        const uint64_t bits = wave_reduce(found ? 1ull << (v & 63) : 0ull, 0ull, [](uint64_t x, uint64_t y) { return x | y; });
        if (ln == 0) atomicOr((unsigned long long *)&T.fnext[v0 >> 6], (unsigned long long)bits);
        if (found) team_found<true>(a, T, t, v, id, dv);
    }
}

// A team phase: rounds from L on, by this member of the team, while they stay
// small (kWhole, a graph the team runs whole: to the end). The state it leaves
// is what a grid round expects: frontier L as a bitmap, its counts in E; after
// the last round, what the epilogue leaves but for the counters. Returns
// false when a wait expired; E.more: rounds are left. At most `cap` rounds;
// `t_start` is the trace's time 0. `level1`: frontier L is round 0's, its levels
// (1) not yet written. `order` (from level 0): receives the reached
// vertices level by level, loff[l] the first position of level l.
template <int BS, bool kWhole>
__device__ __forceinline__ bool bfs_team_phase(const BfsArgs &a, TeamLds &t, TeamBits *front, uint64_t *s_vis,
                                               uint32_t members,
                                               uint32_t rank, uint32_t &tag, RoundState &S, const RoundCounts &rc,
                                               long long t_start, uint32_t cap, bool level1, TeamEnd &E,
                                               uint32_t *order = nullptr, uint32_t *loff = nullptr)
{
    constexpr int WPB = BS / kWave;
    const uint32_t W = a.g.words;
    const uint32_t tid = rank * BS + threadIdx.x, nthreads = members * BS;
    const bool lead = rank == 0 && threadIdx.x == 0;
    BfsTeam T;
    T.members = members;
    T.rank = rank;
    T.tag = tag;
    T.gwave = rank * WPB + threadIdx.x / kWave;
    T.nwaves = members * WPB;
    T.seg = a.qcap / members;
    T.front = front;
    T.s_vis = s_vis;
    if (kWhole)
        for (uint32_t w = threadIdx.x; w < W; w += BS) T.s_vis[w] = load_team(a.vis + w);
    bool ok = true;
    uint32_t &L = S.L;
    if (kWhole) {
        T.total = rc.count;
    } else if (S.pol.pull_prev || rc.overflow) {
        // no queue: each member gathers its share of the bitmap into its segment
        team_gather(t, a.fbit + (size_t)(L % 3) * W, W, a.queue + (size_t)(L % 3) * a.qcap + (size_t)rank * T.seg, tid,
                    nthreads);
        ok = team_exchange(a.bar, t, members, rank, T.tag, a.abort);
        team_segments(T, t);
    } else {
        T.incl = T.total = rc.qlen;  // the grid's queue is one segment
    }
    const uint32_t limit = team_limit(a.qcap, kTeamPushEdges);
    unsigned long long count = rc.count, scout = rc.scout;
    bool hubs = rc.has_huge;
    uint32_t placed = 0;  // vertices of the levels before L
    if (!kWhole && level1) {
        const uint32_t *q1 = a.queue + (size_t)(L % 3) * a.qcap;
        for (uint32_t i = tid; i < T.total; i += nthreads) a.level[caller_id(a, load_team(q1 + i))] = (int32_t)L;
    }
    // a phase of narrow rounds keeps no bitmaps and leaves all three clear meanwhile
    if (!kWhole)
        for (uint32_t w = tid; w < W; w += nthreads) {
            a.fbit[(size_t)(L % 3) * W + w] = 0;
            a.fbit[(size_t)((L + 2) % 3) * W + w] = 0;
        }
    bool more = ok;
    for (uint32_t r = 0; more && r < cap; r++) {
        const bool pull = S.next(count, scout);
        if (lead) write_trace(a.trace, L, pull, count, scout, t_start);
        T.L = L;
        T.qin = a.queue + (size_t)(L % 3) * a.qcap;
        T.qout = a.queue + (size_t)((L + 1) % 3) * a.qcap + (size_t)rank * T.seg;
        T.fnext = a.fbit + (size_t)((L + 1) % 3) * W;
        if constexpr (kWhole) {
            for (uint32_t w = tid; w < W; w += nthreads) a.fbit[(size_t)((L + 2) % 3) * W + w] = 0;
            for (uint32_t w = threadIdx.x; w < W; w += BS) {
                const uint64_t x = load_team(a.fbit + (size_t)(L % 3) * W + w);
                T.front->word[w] = x;
                T.s_vis[w] |= x;
            }
            __syncthreads();
            if (!pull || order) team_bits_count(*T.front, W);
            if (order) {
                for (uint32_t w = tid; w < W; w += nthreads) {
                    uint32_t at = placed + T.front->before[w];
                    for (uint64_t x = T.front->word[w]; x; x &= x - 1) order[at++] = w * 64 + (uint32_t)first_lane(x);
                }
                if (lead) loff[L] = placed;
                placed += T.total;
                if (lead) loff[L + 1] = placed;
            }
            if (pull) team_pull(a, T, t);
            else team_push<true>(a, T, t, hubs);
        } else {
            team_push<false>(a, T, t, false);
        }
        S.pol.pull_prev = pull;
        L++;
        ok = team_exchange(a.bar, t, members, rank, T.tag, a.abort);
        if (!ok) break;
        const uint64_t w = team_segments(T, t);
        count = T.total;
        scout = wave_sum_u64(w & 0xFFFFFFFFu);
        hubs = ballot((w >> kTeamFlagShift) & 1) != 0;
        more = count != 0 && !(a.max_rounds && L >= a.max_rounds);
        if (more && !kWhole) {
            DirectionPolicy p = S.pol;
            if (hubs || count > limit || scout > limit || p.next(L, count, scout)) break;
        }
    }
    tag = T.tag;
    if (!ok) return false;
    uint64_t *fl = a.fbit + (size_t)(L % 3) * W;
    if (kWhole) {
        // the last round: bitmaps are left clear for the next query
        for (uint32_t w = tid; w < 3 * W; w += nthreads) a.fbit[w] = 0;
    } else if (more) {
        const uint32_t own = (uint32_t)((t.slot[rank] >> kTeamCountShift) & kTeamCountMask);
        const uint32_t *q = a.queue + (size_t)(L % 3) * a.qcap + (size_t)rank * T.seg;
        for (uint32_t i = threadIdx.x; i < own; i += BS) {
            const uint32_t u = load_team(q + i);
            atomicOr((unsigned long long *)&fl[u >> 6], 1ull << (u & 63));
        }
    }
    E.count = count;
    E.scout = scout;
    E.hubs = hubs;
    E.more = more;
    return true;
}

// The whole query on the team, for a graph it runs whole: the other blocks
// return after the census, so no grid barrier is taken. Every state the next
// query expects is left as the grid's own path leaves it. A query by grid
// rounds and by this path: RMAT graphs of 4096 vertices 56 and 37 us, of 8001 62
// and 41, of 16001 67 and 51, of 32001 70 and 84 (one XCD's caches and CUs
// no longer suffice), so the line lies at 16384 vertices.
// `t` is reset here; members, rank (~0: none) and tag are this block's place
// for what follows the traversal; `order`, `loff`: see bfs_team_phase.
template <int BS>
__device__ __forceinline__ bool bfs_whole(const BfsArgs &a, TeamLds &t, uint32_t xcc, BarState &gen, uint32_t &members,
                                          uint32_t &rank, uint32_t &tag, uint32_t *order = nullptr,
                                          uint32_t *loff = nullptr)
{
    __shared__ uint32_t s_ok;
    __shared__ TeamBits s_front;
    __shared__ uint64_t s_vis[kTeamWords];
    const long long t_start = wall_clock64();
    const DevGraph &g = a.g;
    const uint32_t W = g.words, src = a.source;
    const uint32_t sdeg = g.row[src + 1] - g.row[src];
    tag = 0;
    if (threadIdx.x == 0) t.reset();
    if (threadIdx.x == 0) s_ok = bar_census(a.bar, xcc, gen, a.abort);
    team_place(xcc, gen, members, rank);
    RoundState S{{a.alpha, a.beta, a.total_workload0, g.n, a.force}, 0, 0, 0, 0};
    bool ok = s_ok != 0u;
    if (ok && rank == ~0u) return true;
    if (ok) {
        const uint32_t tid = rank * BS + threadIdx.x, nthreads = members * BS;
        for (uint32_t i = tid; i < g.n; i += nthreads) a.level[i] = i == a.source_id ? 0 : -1;
        for (uint32_t w = tid; w < W; w += nthreads) {
            const uint64_t sb = w == (src >> 6) ? 1ull << (src & 63) : 0ull;
            const uint64_t inert = g.inert ? g.inert[w] : 0ull;
            a.vis[w] = inert | sb;
            a.vis_idle[w] = inert;
            a.fbit[w] = sb;
            a.fbit[(size_t)W + w] = 0;
            a.fbit[2 * (size_t)W + w] = 0;
        }
        ok = team_exchange(a.bar, t, members, rank, tag, a.abort);
    }
    if (ok) {
        const RoundCounts rc{1, sdeg, 1, false, sdeg > kHugeDegree};
        TeamEnd E{};
        ok = bfs_team_phase<BS, true>(a, t, &s_front, s_vis, members, rank, tag, S, rc, t_start, ~0u, false, E, order, loff);
        // (the other blocks read no counters)
        if (ok && rank == 0)
            for (int i = 0; i < 3; i++) clear_ctr(&a.ctr[i]);
    }
    // (after a failed census no block's place is known: block 0 reports)
    if (!s_ok) rank = blockIdx.x ? ~0u : 0u;
    if (rank == 0 && threadIdx.x == 0)
        write_final(a.trace, a.stats, S.L, S.pushes, S.pulls, S.ptrace, ok, t_start);
    return ok;
}

#if SG_BFS_WAVES
#define SG_BFS_BOUNDS(BS) __launch_bounds__(BS, SG_BFS_WAVES)
#else
#define SG_BFS_BOUNDS(BS) __launch_bounds__(BS)
#endif

// One BFS query over the `nblocks` blocks of a persistent grid (this block
// is number `brank` of them): the whole launch, or the blocks one XCD holds
// when a launch serves one query per XCD. `gen` is the block's barrier state
// for a.bar (from bar_begin or the caller's census), advanced by every
// barrier. Returns false when a bounded wait expired (the run then stopped).
// kStage: push rounds stage hub neighbour lists in LDS (the engine option
// stage_hubs; a separate instantiation, so the default path keeps its
// register budget).
// kTeamOk: rounds with little work may run on the team (a.team; needs `gen`
// from bar_begin<true> on a.bar, whose first barrier takes the census).
// kLeave: nothing follows the traversal, so blocks may return before every
// block has seen its end. kEven: the graph is not skewed (a.team 2 or 0). team, team_tag, team_phase: the caller's own team
// state, when its team goes on after the traversal.
template <int BS, bool kStage = false, bool kTeamOk = false, bool kLeave = false, bool kEven = false>
__device__ __forceinline__ bool bfs_run(const BfsArgs &a, uint32_t brank, uint32_t nblocks, uint32_t xcc,
                                        BarState &gen, TeamLds *team = nullptr, uint32_t *team_tag = nullptr,
                                        uint32_t *team_phase = nullptr)
{
    constexpr int WPB = BS / kWave;
    constexpr uint32_t kLdsQ = 8u * BS;
    const DevGraph &g = a.g;
    const uint32_t n = g.n, W = g.words;
    const uint32_t gtid = brank * BS + threadIdx.x;
    const uint32_t nthreads = nblocks * BS;
    const uint32_t gwave = brank * WPB + threadIdx.x / kWave;
    const uint32_t nwaves = nblocks * WPB;
    const int ln = lane();
    const long long t_start = wall_clock64();

    __shared__ unsigned long long s_red[2][WPB];
    __shared__ unsigned long long s_lvl[5];
    __shared__ uint32_t s_q[kLdsQ];
    __shared__ uint32_t s_qn, s_flush[2];
    // hub round: the block's member chunks (first edge, end) and their staged heads
    __shared__ uint2 s_hc[kStage ? kHubList : 1];
    __shared__ uint32_t s_he[kStage ? kStageChunks * kHugeChunk : 1];
    __shared__ uint32_t s_hn;
    __shared__ TeamLds s_own;
    TeamLds &s_t = team ? *team : s_own;
    uint32_t phase0 = 0, tag0 = 0;
    uint32_t &phase = team_phase ? *team_phase : phase0, &tag = team_tag ? *team_tag : tag0;
    if (kTeamOk && threadIdx.x == 0) s_t.reset();

    // ---- prologue: reset the levels (caller order) and seed the source.
    // The previous query left the frontier bitmaps and counters zeroed, and
    // visited filters alternate between two buffers (the idle one is reset
    // here for the next query), so with a narrow source block 0 expands it
    // (round 0) while the other blocks reset, and one barrier ends both.
    const uint32_t src = a.source;
    const uint32_t sbeg = g.row[src], sdeg = g.row[src + 1] - sbeg;
    const uint64_t sbit = 1ull << (src & 63);
    if (kTeamOk && gtid == 0) team_clock_set(a.bar, t_start);
    for (uint32_t i = gtid; i < n; i += nthreads) a.level[i] = (i == a.source_id) ? 0 : -1;
    for (uint32_t w = gtid; w < W; w += nthreads) a.vis_idle[w] = g.inert ? g.inert[w] : 0ull;
    RoundState S{{a.alpha, a.beta, a.total_workload0, n, a.force}, 0, 0, 0, 0};  // replicated in every block
    uint32_t &L = S.L;
    const bool local0 = !a.full_init && a.force != 1 && sdeg <= kLocalRound0;
    if (!local0) {
        // state of unknown content (first query, other work since), a wide
        // source or forced pull: reset everything, round 0 over the grid
        for (uint32_t w = gtid; w < W; w += nthreads) {
            const uint64_t sb = (w == (src >> 6)) ? sbit : 0ull;
            a.vis[w] = (g.inert ? g.inert[w] : 0ull) | sb;
            a.fbit[w] = sb;                    // frontier 0
            a.fbit[(size_t)W + w] = 0;         // frontier 1, built by round 0
            a.fbit[2 * (size_t)W + w] = 0;
        }
        if (brank == 0) {
            clear_ctr(&a.ctr[0]);
            clear_ctr(&a.ctr[1]);
            clear_ctr(&a.ctr[2]);
            block_sync_global();
            if (threadIdx.x == 0) {
                a.queue[0] = src;
                a.ctr[0].qlen = 1;
                a.ctr[0].has_huge = sdeg > kHugeDegree;
                a.ctr[0].stripe[0].scout = sdeg;
                a.ctr[0].stripe[0].count = 1;
            }
        }
    } else if (brank == 0) {
        // round 0 without its levels: other blocks are still resetting the
        // level array, so round 1 writes level 1 for the queue it reads
        if (threadIdx.x == 0) {
            atomicOr((unsigned long long *)&a.vis[src >> 6], (unsigned long long)sbit);
            s_qn = 0;
        }
        block_sync_global();
        Round R;
        R.a = &a;
        R.L = 0;
        R.fcur = nullptr;
        R.fnext = a.fbit + (size_t)W;
        R.S = Stager{a.queue + (size_t)a.qcap, a.qcap, &a.ctr[1], s_q, &s_qn, kLdsQ};
        R.scout = 0;
        R.count = 0;
        R.huge = false;
        R.levels = false;
        for (uint32_t e0 = (threadIdx.x / kWave) * kWave; e0 < sdeg; e0 += WPB * kWave) {
            const uint32_t e = e0 + (uint32_t)ln;
            const bool act = e < sdeg;
            push_visit(R, act, act ? g.col[sbeg + e] : 0u);
        }
        flush_stage(R.S, s_flush);
        publish_counts<WPB>(&a.ctr[1], R.scout, R.count, R.huge, s_red);
    }
    bool ok = grid_sync(a.bar, xcc, gen, a.abort);
    if (local0) {
        S.next(1, sdeg);  // push, as every round 0
        if (gtid == 0) write_trace(a.trace, 0, false, 1, sdeg, t_start);
        L = 1;
    }

    // the grid's rounds use the counter slots in turn; the team's use none, and
    // after a phase the counts come with its note
    uint32_t slot = L;
    __shared__ uint32_t s_prev;  // (kEven) see team_stays()
    if (kEven && threadIdx.x == 0) s_prev = 0;
    bool noted = false;
    while (ok) {
        if (!noted) read_counts(&a.ctr[slot % 3], s_lvl);
        if (threadIdx.x == 0) s_qn = 0;
        __syncthreads();
        const RoundCounts rc = unpack_counts(s_lvl, a.qcap);
        const uint32_t prev = kEven ? s_prev : 0u;
        __syncthreads();
        const bool last = rc.count == 0 || (a.max_rounds && L >= a.max_rounds);
        const bool team_phase_next = kTeamOk && !last && bfs_team_fits<kLeave, kEven>(a, S, rc, prev);
        noted = false;
        if (kEven && threadIdx.x == 0) s_prev = team_phase_next ? ~0u : (uint32_t)rc.count;
        const bool level1 = L == 1 && local0;
        if (level1 && !team_phase_next) {
            // the source's out-neighbours found by block 0 (at most
            // kLocalRound0, so the queue holds them all); a team's rounds
            // would overwrite the queue under a block that is late here, so
            // before a phase its members write them
            const uint32_t *q1 = a.queue + (size_t)a.qcap;
            for (uint32_t i = gtid; i < rc.qlen; i += nthreads) a.level[caller_id(a, q1[i])] = 1;
        }
        if (last) break;

        if (team_phase_next) {
            uint32_t members, rank;
            team_place(xcc, gen, members, rank);
            TeamEnd E{};
            if (rank != ~0u) {
                // a failed wait set the abort flag, which ends the others' wait
                const long long t0 = rank == 0 && threadIdx.x == 0 ? team_clock(a.bar) : 0ll;
                ok = bfs_team_phase<BS, false>(a, s_t, nullptr, nullptr, members, rank, tag, S, rc, t0, kTeamRounds, level1,
                                               E);
                if (!ok) break;
                if (kLeave && !E.more && rank == 0 && threadIdx.x == 0)
                    write_final(a.trace, a.stats, L, S.pushes, S.pulls, S.ptrace, true, t0);
            }
            ok = team_rejoin<kLeave>(a.bar, xcc, gen, a.abort, phase++, rank, S, E, s_lvl);
            if (ok && E.left) {
                // every block has read the counters: leave them clear for the next query
                if (E.closed)
                    for (int i = 0; i < 3; i++) clear_ctr(&a.ctr[i]);
                return true;
            }
            noted = true;
            continue;
        }

        const bool pull = S.next(rc.count, rc.scout);
        if (gtid == 0) write_trace(a.trace, L, pull, rc.count, rc.scout, t_start);
        if (brank == 0) clear_ctr(&a.ctr[(slot + 2) % 3]);

        Round R;
        R.a = &a;
        R.L = (int32_t)L;
        R.fcur = a.fbit + (size_t)(L % 3) * W;
        R.fnext = a.fbit + (size_t)((L + 1) % 3) * W;
        {
            // frontier L-1 is no longer read: clear its bitmap for round L+1
            uint64_t *fclr = a.fbit + (size_t)((L + 2) % 3) * W;
            for (uint32_t w = gtid; w < W; w += nthreads) fclr[w] = 0;
        }
        R.S = Stager{a.queue + (size_t)((L + 1) % 3) * a.qcap, a.qcap, &a.ctr[(slot + 1) % 3], s_q, &s_qn, kLdsQ};
        R.scout = 0;
        R.count = 0;
        R.huge = false;
        R.even = kEven;
        const uint32_t *qin = a.queue + (size_t)(L % 3) * a.qcap;

        if (!pull) {
            // (1) high-degree frontier vertices through the static chunk list.
            //     With kStage their neighbour lists are staged in LDS
            //     (the reference's CTA-level expansion of large vertices,
            //     cta_scheduler_hybrid.cuh:86-142): thread t of block b
            //     checks descriptors k * nblocks * BS + t * nblocks + b (the
            //     chunks of one hub land in different blocks) and lists the
            //     chunks whose vertex is in the frontier (first edge, end),
            //     up to kHubList at a time; the block then loads their heads
            //     into LDS, kStageChunks chunks per pass with every thread's
            //     loads in flight together, and its waves expand one staged
            //     chunk per step.
            const uint32_t nhuge = rc.has_huge && !a.lb_push_none ? g.nhuge : 0u;
            const uint32_t per = !kStage ? 0u : (nhuge + nblocks * BS - 1) / (nblocks * BS);  // descriptors per thread
            for (uint32_t k0 = 0; k0 < per;) {
                if (threadIdx.x == 0) s_hn = 0;
                __syncthreads();
                // each pass lists at most kHubList chunks: BS threads x kHubList / BS descriptors
                const uint32_t k1 = min(per, k0 + kHubList / BS);
                for (uint32_t k = k0; k < k1; k++) {
                    const uint32_t c = k * nblocks * BS + threadIdx.x * nblocks + brank;
                    if (c < nhuge) {
                        const uint2 dsc = g.huge[c];
                        const uint32_t end = g.huge_end[c];
                        if (in_frontier(R, dsc.x)) s_hc[atomicAdd(&s_hn, 1u)] = make_uint2(dsc.y, end);
                    }
                }
                k0 = k1;
                __syncthreads();
                const uint32_t nm = s_hn;
                for (uint32_t m0 = 0; m0 < nm; m0 += kStageChunks) {
                    const uint32_t mc = min(kStageChunks, nm - m0);
                    for (uint32_t i = threadIdx.x; i < mc * kHugeChunk; i += BS) {
                        const uint2 ch = s_hc[m0 + i / kHugeChunk];
                        const uint32_t e = ch.x + i % kHugeChunk;
                        s_he[i] = e < ch.y ? g.col[e] : kNoHead;
                    }
                    __syncthreads();
                    for (uint32_t q = threadIdx.x / kWave; q < mc; q += WPB) {
                        const uint32_t v = s_he[q * kHugeChunk + (uint32_t)ln];
                        push_visit(R, v != kNoHead, v != kNoHead ? v : 0u);
                    }
                    __syncthreads();
                }
                __syncthreads();  // every thread has read the count before it is reset
            }
            //     Otherwise (the default: on RMAT-22 staging measured 6 %
            //     slower for the whole query, its block barriers outweighing
            //     the overlapped loads) lane ln of wave gw takes chunk
            //     base + ln * nwaves + gw, so the chunks of one hub land on
            //     different waves, and each wave expands its member chunks
            //     one after another.
            for (uint32_t base = 0; !kStage && base < nhuge; base += nwaves * kWave) {
                const uint32_t c = base + (uint32_t)ln * nwaves + gwave;
                uint2 dsc = make_uint2(0u, 0u);
                uint32_t end = 0;
                bool mem = false;
                if (c < nhuge) {
                    dsc = g.huge[c];
                    end = g.huge_end[c];
                    mem = in_frontier(R, dsc.x);
                }
                uint64_t mm = ballot(mem);
                while (mm) {
                    const int t = first_lane(mm);
                    mm &= mm - 1;
                    const uint32_t beg = lane_value(dsc.y, t), stop = lane_value(end, t);
                    for (uint32_t e0 = beg; e0 < stop; e0 += kWave) {
                        const uint32_t e = e0 + ln;
                        const bool act = e < stop;
                        push_visit(R, act, act ? g.col[e] : 0u);
                    }
                }
            }
            // (2) the rest of the frontier: from the queue after a push round,
            //     from the bitmap after a pull round or if the queue overflowed.
            if (S.pol.pull_prev || rc.overflow) {
                // words dealt round-robin: in a degree-ordered graph adjacent
                // words hold vertices of similar degree
                for (uint32_t wb = 0; wb < W; wb += nwaves * kWave) {
                    const uint32_t w = wb + (uint32_t)ln * nwaves + gwave;
                    const uint64_t fl = w < W ? R.fcur[w] : 0ull;
                    wave_word_vertices(fl, w, [&](bool valid, uint32_t u) {
                        if (a.lb_push_none) push_expand_serial(R, valid, u);
                        else push_expand(R, valid, u);
                    });
                }
            } else {
                // entries dealt round-robin, lane ln of wave gw taking entry
                // base + ln * nwaves + gw: a short queue puts one vertex on each
                // of many waves, and no wave gets a run of entries staged
                // together (neighbours of one hub)
                for (uint32_t i0 = 0; i0 < rc.qlen; i0 += nwaves * kWave) {
                    const uint32_t i = i0 + (uint32_t)ln * nwaves + gwave;
                    const bool valid = i < rc.qlen;
                    if (!ballot(valid)) break;
                    if (a.lb_push_none) push_expand_serial(R, valid, valid ? qin[i] : 0u);
                    else push_expand(R, valid, valid ? qin[i] : 0u);
                }
            }
        } else {
            // Pull: sweep this wave's words, skipping ones the filter marks
            // full. Words are dealt round-robin (lane ln of wave gw takes word
            // base + ln * nwaves + gw): unreached high-in-degree vertices walk
            // long in-edge lists, and they cluster at low ids (RMAT,
            // degree-ordered graphs).
            for (uint32_t wb = 0; wb < W; wb += nwaves * kWave) {
                const uint32_t wl = wb + (uint32_t)ln * nwaves + gwave;
                const uint64_t vl = wl < W ? a.vis[wl] : ~0ull;
                if (wl < W && vl == ~0ull) R.fnext[wl] = 0;
                uint64_t todo = ballot(vl != ~0ull);
                if (a.lb_pull_none) {
                    while (todo) {
                        const int t = first_lane(todo);
                        todo &= todo - 1;
                        pull_word_serial(R, wb + (uint32_t)t * nwaves + gwave, lane_value(vl, t));
                    }
                }
                while (todo) {
                    constexpr int G = kPullGroup;
                    uint32_t wg[G];
                    uint64_t vwg[G];
                    int ng = 0;
#pragma unroll
                    for (int i = 0; i < G; i++) {
                        wg[i] = wb;
                        vwg[i] = ~0ull;
                        if (todo) {
                            const int t = first_lane(todo);
                            todo &= todo - 1;
                            wg[i] = wb + (uint32_t)t * nwaves + gwave;
                            vwg[i] = lane_value(vl, t);
                            ng++;
                        }
                    }
                    pull_group<G>(R, wg, vwg, ng);
                }
            }
        }
        // counters first: their atomics are then in flight while the queue
        // flush waits for its position
        publish_counts<WPB>(R.S.nxt, R.scout, R.count, R.huge, s_red);
        flush_stage(R.S, s_flush);
        S.pol.pull_prev = pull;
        L++;
        slot++;
        ok = grid_sync(a.bar, xcc, gen, a.abort);
    }

    // ---- epilogue: every block left the loop after the same barrier, which
    // made the last round's levels visible. Zero the frontier bitmaps and
    // counters for the next query.
    if (ok) {
        for (uint32_t w = gtid; w < 3 * W; w += nthreads) a.fbit[w] = 0;
        if (brank == 0) {
            clear_ctr(&a.ctr[0]);
            clear_ctr(&a.ctr[1]);
            clear_ctr(&a.ctr[2]);
        }
    }
    if (gtid == 0) write_final(a.trace, a.stats, L, S.pushes, S.pulls, S.ptrace, ok, t_start);
    return ok;
}

}  // namespace bfsk
}  // namespace
