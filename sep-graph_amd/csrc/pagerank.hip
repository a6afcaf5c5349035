// PageRank as persistent kernels: a topology-driven pull (power iteration)
// and a data-driven residual propagation that switches between push and pull
// per round.
//
// Reference path: samples/hybrid_pr/hybrid_pr.cu:26-125 (the PageRank app:
// residual push, AccumulateBuffer with float atomicAdd) driven by
// RunSyncPullTD (include/framework/algo_variants.cuh:753-823, topology-driven
// pull over the CSC) or RunAsyncPushDD (algo_variants.cuh:133-203, worklist of
// vertices whose residual crossed the threshold, hybrid_pr.cu:66-110).
//
// The ranks computed here are the normalised PageRank with uniform teleport
// and uniform redistribution of dangling mass,
//     x = (1-d)/n + d (P^T x + (sum of x over dangling vertices)/n),
// stored as FP32. Sums are compensated FP32 (hi + lo): in-edge sums and the
// dangling mass, in the residual mode the unnormalised ranks, the residuals
// (each atomic addition's rounding error, recomputed by the adding lane, goes
// to a second FP32 array) and the normalising sum; only the L1 residual (pull)
// and the residual mass absorbed at the end (DD) are reduced in FP64. In the
// pull mode every reduction runs in a fixed order for a given grid, so repeated
// runs give identical bits. (FP64 sums, two instructions per in-edge instead of
// seven: RMAT-21 pull 1750 us and 1778, 100 003 vertices DD 2151 and 2182.)
//
// Pull TD: one lane per vertex sums x[u]/outdeg(u) (kept as an FP32 array
// `contrib`, ping-ponged between iterations) over its in-edges, reading them
// row by row from the graph's sliced in-edge layout (a lane's own entries,
// in order; without that layout, the wave walks the concatenated in-edge
// lists 64 edges per step with a segmented scan). Vertices with in-degree
// above kPullHubDegree are summed per 256-edge chunk; a hub of one chunk is
// finished with it, the others after a grid barrier, eight lanes per hub.
//
// Residual DD: solves the unnormalised system y = (1-d)/n + d P^T y by
// residual propagation (dangling mass leaks) and normalises y at the end; for
// uniform teleport this is the same ranking vector, x = y / |y|_1. A round
// activates every vertex whose residual reached theta = tol (1-d) / n (the
// rounds' worklist holds vertices whose residual crossed theta), moves the
// residual into y and spreads d r / outdeg along out-edges: with FP32 atomics
// when the active out-degree is small (push), or by a gather over in-edges
// when it exceeds m / alpha (pull, which activates for the next round in the
// same pass).
#include "frontier.hpp"

using namespace sg;

namespace {

// ------------------------------------------- compensated FP32 accumulation
// A sum kept as hi + lo, where lo collects the rounding error of every
// addition into hi (TwoSum, Knuth: exact, and without the comparison of
// Neumaier's form): FP32 storage and arithmetic with an error close to one
// rounding of the final sum.
struct CSum {
    float hi, lo;
};

__device__ __forceinline__ void csum_add(CSum &a, float x)
{
    const float s = a.hi + x;
    const float b = s - a.hi;
    const float t = (a.hi - (s - b)) + (x - b);
    a.hi = s;
    a.lo += t;
}

// a then b (the order fixes the rounding)
__device__ __forceinline__ CSum csum_merge(CSum a, const CSum &b)
{
    csum_add(a, b.hi);
    a.lo += b.lo;
    return a;
}

__device__ __forceinline__ float csum_value(const CSum &a) { return a.hi + a.lo; }

// The same sum with its value in hi and what that rounds off in lo (TwoSum).
__device__ __forceinline__ CSum csum_settle(const CSum &a)
{
    CSum s{a.hi, 0.f};
    csum_add(s, a.lo);
    return s;
}

// Wave sum, merged lower lanes first in a fixed order; every lane has the
// same bits.
__device__ __forceinline__ CSum wave_csum(CSum a)
{
    return wave_reduce(a, CSum{0.f, 0.f}, [](const CSum &x, const CSum &y) { return csum_merge(x, y); });
}

// Segmented inclusive compensated sum (owners non-decreasing along the wave).
__device__ __forceinline__ CSum seg_csum(CSum s, int k)
{
    return wave_seg_scan(s, (uint32_t)k, [](const CSum &x, const CSum &y) { return csum_merge(x, y); });
}

// Per-block partials of the pull iteration: the L1 residual in FP64 and the
// dangling mass as a compensated FP32 sum (16 bytes, the size of a double2).
struct PrPart {
    double res;
    float dhi, dlo;
};
static_assert(sizeof(PrPart) == sizeof(double2), "PrPart shares the partial-sum area with double2 partials");
static_assert(sizeof(CSum) == 8, "hub chunk sums are 8 bytes");

// Block sums of (residual, dangling) in a fixed order; valid in thread 0.
template <int WPB>
__device__ __forceinline__ PrPart block_part(double res, CSum dang, PrPart *s_red)
{
    res = wave_sum_f64(res);
    dang = wave_csum(dang);
    const int wid = threadIdx.x / kWave;
    if (lane() == 0) s_red[wid] = PrPart{res, dang.hi, dang.lo};
    __syncthreads();
    PrPart t{0.0, 0.f, 0.f};
    if (threadIdx.x == 0) {
        CSum c{0.f, 0.f};
        for (int i = 0; i < WPB; i++) {
            t.res += s_red[i].res;
            c = csum_merge(c, CSum{s_red[i].dhi, s_red[i].dlo});
        }
        t.dhi = c.hi;
        t.dlo = c.lo;
    }
    __syncthreads();
    return t;
}

// Sum of the per-block partials in a fixed order, returned to every thread.
template <int BS>
__device__ __forceinline__ PrPart grid_part(const PrPart *part, uint32_t nblocks, PrPart *s_red, PrPart *s_out)
{
    double res = 0.0;
    CSum dang{0.f, 0.f};
    for (uint32_t i = threadIdx.x; i < nblocks; i += BS) {
        const PrPart q = part[i];
        res += q.res;
        dang = csum_merge(dang, CSum{q.dhi, q.dlo});
    }
    const PrPart t = block_part<BS / kWave>(res, dang, s_red);
    if (threadIdx.x == 0) *s_out = t;
    __syncthreads();
    const PrPart r = *s_out;
    __syncthreads();
    return r;
}

// Sum over the in-edges [b, e) of each lane's vertex of val(edge) as a
// compensated FP32 sum, the wave walking the concatenated lists 4 x 64
// edges per iteration (all of an iteration's loads issued before its
// reductions); each 64-edge sub-step reduces its segments in a fixed order,
// so the result is deterministic.
template <typename F>
__device__ __forceinline__ CSum wave_gather_csum(uint32_t b, uint32_t e, F val)
{
    constexpr int Q = 4;
    const int ln = lane();
    CSum acc{0.f, 0.f};
    for (;;) {
        const uint32_t r = e - b;
        const uint32_t incl = wave_incl_scan(r);
        const uint32_t total = lane_value(incl, kWave - 1);
        if (total == 0) break;
        const uint32_t excl = incl - r;
        int k[Q];
        float cand[Q];
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const uint32_t j = (uint32_t)(q * kWave + ln);
            k[q] = owner_lane(incl, j < total ? j : total - 1);
            const uint32_t bk = shfl(b, k[q]), xk = shfl(excl, k[q]);
            cand[q] = j < total ? val(bk + (j - xk)) : 0.f;
        }
        const uint32_t span = min(total, (uint32_t)(Q * kWave));
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const uint32_t s0 = (uint32_t)(q * kWave);
            if (s0 >= span) break;  // wave-uniform
            const CSum s = seg_csum(CSum{cand[q], 0.f}, k[q]);
            const uint32_t lo = min(max(excl, s0), s0 + kWave), hi = min(max(incl, s0), min(span, s0 + kWave));
            const int at = (int)(hi > s0 ? hi - 1 - s0 : 0);
            const CSum seg{__shfl(s.hi, at, kWave), __shfl(s.lo, at, kWave)};
            if (hi > lo) acc = csum_merge(acc, seg);
        }
        b += min(incl, span) - min(excl, span);
    }
    return acc;
}

// ------------------------------------------------------------ pull TD kernel

// The sum over each row of 16 lanes, in the row's first lane in a fixed order.
__device__ __forceinline__ CSum row_csum(CSum x)
{
    const CSum none{0.f, 0.f};
    x = csum_merge(x, dpp<kDppRowRor + 8>(none, x));
    x = csum_merge(x, dpp<kDppRowRor + 4>(none, x));
    x = csum_merge(x, dpp<kDppRowRor + 2>(none, x));
    x = csum_merge(x, dpp<kDppRowRor + 1>(none, x));
    return x;
}

// Four wave sums together: lane l gets that of s[l % 4]. Halves of the wave,
// then rows of 16 lanes, trade places between two sums, so that three merges
// leave one sum per row and four more finish them, where four scans take 24.
__device__ __forceinline__ CSum wave_csum4(const CSum (&s)[4])
{
    auto fold = [](CSum a, CSum b, bool half) {
        uint32_t x[2], y[2];
        __builtin_memcpy(x, &a, 8);
        __builtin_memcpy(y, &b, 8);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const auto r = half ? __builtin_amdgcn_permlane32_swap(x[i], y[i], false, false)
                                : __builtin_amdgcn_permlane16_swap(x[i], y[i], false, false);
            x[i] = r[0];
            y[i] = r[1];
        }
        __builtin_memcpy(&a, x, 8);
        __builtin_memcpy(&b, y, 8);
        return csum_merge(a, b);
    };
    // rows of (0, 2): 0 0 2 2; of (1, 3): 1 1 3 3; of both: 0 1 2 3
    const CSum t = row_csum(fold(fold(s[0], s[2], true), fold(s[1], s[3], true), false));
    const int from = (lane() & 3) * 16;
    return CSum{shfl(t.hi, from), shfl(t.lo, from)};
}

// ---------------------------------------------- sums over every in-edge list
// Both kernels sum one FP32 value per source over all in-edges. The values of
// the lowest ids (in a degree-ordered graph the sources of most in-edges) are
// copied to LDS before a pass (they are read-only until the next barrier), and
// the gather reads them there instead of sending one L2 request per in-edge.
constexpr uint32_t kNoEdge = 0xFFFFFFFFu;

// Floats from one row of values to the next: 16-byte aligned rows.
__host__ __device__ constexpr uint64_t contrib_stride(uint32_t n) { return ((uint64_t)n + 3) / 4 * 4; }

// The copy: KF floats per thread, 16 bytes a lane straight from memory into
// LDS, so that it takes no registers while other loads of the round are waited
// for. take() starts it (once every wave is done with the last copy), wait()
// and a __syncthreads() end it.
template <int BS, int KF>
struct Staged {
    static constexpr uint32_t kLds = (uint32_t)KF * BS;
    static constexpr int kFill = (int)((kLds / 4 + BS - 1) / BS);
    static __device__ __forceinline__ void take(float *s_cc, const float *cc, uint32_t n)
    {
        const uint32_t have = min(n, kLds);
        const uint32_t wave0 = __builtin_amdgcn_readfirstlane(threadIdx.x & ~(uint32_t)(kWave - 1));
#pragma unroll
        for (int i = 0; i < kFill; i++) {
            if (4 * threadIdx.x < have - min(have, (uint32_t)(4 * i * BS)))
                __builtin_amdgcn_global_load_lds(
                    (__attribute__((address_space(1))) void *)((const float4 *)cc + i * BS + threadIdx.x),
                    (__attribute__((address_space(3))) void *)((float4 *)s_cc + i * BS + wave0), 16, 0, 0);
        }
    }
    static __device__ __forceinline__ void wait() { __builtin_amdgcn_s_waitcnt(0); }
};

// Values of N sources: the loads of those outside LDS are all issued first,
// then every entry reads LDS (s_cc[K], a zero, if it has no place there), so
// no entry waits for the one before it.
template <uint32_t K>
struct Gather {
    const float *cc, *s_cc;
    uint32_t n;
    template <int N>
    __device__ __forceinline__ void get(const uint32_t (&u)[N], float (&c)[N]) const
    {
        const uint32_t ncold = n > K ? n - K : 0u;
#pragma unroll
        for (int q = 0; q < N; q++) {
            c[q] = 0.f;
            if (u[q] - K < ncold) c[q] = cc[u[q]];
        }
#pragma unroll
        for (int q = 0; q < N; q++) c[q] += s_cc[min(u[q], K)];
    }
    __device__ __forceinline__ float one(uint32_t u) const { return u < min(n, K) ? s_cc[u] : cc[u]; }
};

// The bounds a wave starts every pass with: of up to 64 in-hub chunks, of up
// to 64 words of the sliced layout and of its first in-hubs. They never change, so they are read once per
// run, not in every round from caches that the barrier before it emptied (RMAT
// graphs, 17 iterations: 400 001 vertices 477 -> 462 us, 8001 213 -> 209).
struct Bounds {
    uint32_t hv, beg, len;  // chunk gwave + lane * nwaves: hub, first in-edge, in-edges
    bool one;               // the chunk is all of the hub
    uint32_t off, nrow;     // word gwave + lane * nwaves
    uint32_t at, chunks, v; // hub gwave + lane / kHubLanes * nwaves, if of several chunks

    static constexpr uint32_t kHubLanes = 8;

    __device__ __forceinline__ void chunk(const DevGraph &g, uint32_t first, uint32_t nwaves)
    {
        const uint64_t c = first + (uint64_t)lane() * nwaves;
        hv = beg = len = 0;
        one = false;
        if (c < g.nhugein) {
            const uint2 dsc = g.hugein[c];
            hv = dsc.x;
            beg = dsc.y;
            const uint32_t b = g.cstart[hv], e = g.cstart[hv + 1];
            len = min(e - beg, kPullChunk);
            one = e - b <= kPullChunk;
        }
    }
    __device__ __forceinline__ void word(const DevGraph &g, uint32_t first, uint32_t nwaves)
    {
        const uint64_t w = first + (uint64_t)lane() * nwaves;
        off = nrow = 0;
        if (g.sell_src && w < g.words) {
            off = g.sell_off[w];
            nrow = (g.sell_off[w + 1] - off) / kWave;
        }
    }
    __device__ __forceinline__ void hub(const DevGraph &g, uint32_t first, uint32_t nwaves)
    {
        const uint64_t h = first + (uint64_t)(lane() / kHubLanes) * nwaves;
        at = chunks = v = 0;
        if (h < g.nhubin) {
            const uint2 d = g.hubin[h];
            at = d.x;
            chunks = d.y;
            if (d.y > 1) v = g.hugein[d.x].x;
        }
    }
    __device__ __forceinline__ Bounds(const DevGraph &g, uint32_t gwave, uint32_t nwaves)
    {
        chunk(g, gwave, nwaves);
        word(g, gwave, nwaves);
        hub(g, gwave, nwaves);
    }
};

// Chunk sums of the in-hubs, dealt out one by one. A lane holds one chunk's
// bounds and, in the end, its sum; the wave adds kQ chunks together, the next
// kQ chunks' in-edges in flight meanwhile. pre(v): what the hub needs in the
// end, loaded with the bounds (false: no chunk); done(has, c, v, one, own,
// sum), wave-convergent: `one` if chunk c is all of hub v.
template <typename G, typename Pre, typename Done>
__device__ __forceinline__ void hub_chunk_sums(const DevGraph &g, const G &gather, const Bounds &bounds, uint32_t gwave,
                                               uint32_t nwaves, Pre pre, Done done)
{
    constexpr int kQ = 4, kSteps = (int)(kPullChunk / kWave);
    const int ln = lane();
    for (uint32_t first = gwave; first < g.nhugein; first += nwaves * kWave) {
        const uint32_t cnt = min((uint32_t)kWave, (g.nhugein - first + nwaves - 1) / nwaves);
        const uint32_t c = first + (uint32_t)ln * nwaves;
        const bool has = (uint32_t)ln < cnt;
        Bounds bd = bounds;
        if (first != gwave) bd.chunk(g, first, nwaves);
        const uint32_t hv = bd.hv, beg = bd.beg, len = bd.len;
        const bool one = bd.one;
        const auto own = pre(has, hv);
        auto load = [&](uint32_t j, uint32_t (&u)[kQ * kSteps]) {
#pragma unroll
            for (int q = 0; q < kQ; q++) {
                const uint32_t l = lane_value(len, (int)j + q);
                const uint32_t *src = g.csrc + lane_value(beg, (int)j + q);
#pragma unroll
                for (int t = 0; t < kSteps; t++) {
                    const uint32_t k = (uint32_t)(t * kWave + ln);
                    u[q * kSteps + t] = k < l ? src[k] : kNoEdge;
                }
            }
        };
        CSum mine{0.f, 0.f};
        uint32_t u[kQ * kSteps], nu[kQ * kSteps];
        load(0, u);
        for (uint32_t j = 0; j < cnt; j += kQ) {
            if (j + kQ < cnt) load(j + kQ, nu);
            float cv[kQ * kSteps];
            gather.get(u, cv);
            CSum s[kQ];
#pragma unroll
            for (int q = 0; q < kQ; q++) {
                s[q] = CSum{0.f, 0.f};
#pragma unroll
                for (int t = 0; t < kSteps; t++) csum_add(s[q], cv[q * kSteps + t]);
            }
            const CSum t = wave_csum4(s);
            if ((uint32_t)ln / kQ == j / kQ) mine = t;
#pragma unroll
            for (int q = 0; q < kQ * kSteps; q++) u[q] = nu[q];
        }
        done(has, c, hv, one, own, mine);
    }
}

// Sums of every other vertex, a 64-vertex word per wave at a time: from the
// sliced in-edges (each lane sums its own vertex's row entries in order) or,
// without them, by a scheduled walk of the word's lists. What a word's
// vertices need in the end (pre) is loaded one word ahead, its in-edges one
// step ahead. done(has, v, own, sum), wave-convergent. U rows of in-edges at a
// time: the steps of a word are a chain, so as many as there are registers for.
template <uint32_t U, typename G, typename Pre, typename Done>
__device__ __forceinline__ void word_sums(const DevGraph &g, const G &gather, const Bounds &bounds, uint32_t gwave,
                                          uint32_t nwaves, Pre pre, Done done)
{
    const int ln = lane();
    const uint32_t n = g.n, W = g.words;
    if (!g.sell_src) {
        for (uint32_t w = gwave; w < W; w += nwaves) {
            const uint32_t v = w * kWave + ln;
            uint32_t b = 0, e = 0;
            bool has = false;
            if (v < n) {
                b = g.cstart[v];
                e = g.cstart[v + 1];
                has = e - b <= kPullHubDegree;
                if (!has) b = e;
            }
            const auto own = pre(has, v);
            const CSum s = wave_gather_csum(b, e, [&](uint32_t ed) { return gather.one(g.csrc[ed]); });
            done(has, v, own, s);
        }
        return;
    }
    for (uint32_t first = gwave; first < W; first += nwaves * kWave) {
        const uint32_t cnt = min((uint32_t)kWave, (W - first + nwaves - 1) / nwaves);
        Bounds bd = bounds;  // a lane holds one word's rows
        if (first != gwave) bd.word(g, first, nwaves);
        const uint32_t off = bd.off, nrow = bd.nrow;
        auto degree = [&](uint32_t v) { return v < n ? g.cstart[v + 1] - g.cstart[v] : kNoEdge; };
        auto load = [&](uint32_t i, uint32_t j, uint32_t (&u)[U]) {
            const uint32_t rows = lane_value(nrow, (int)i);
            const uint32_t *S = g.sell_src + lane_value(off, (int)i) + ln;
#pragma unroll
            for (uint32_t q = 0; q < U; q++) {
                u[q] = kNoEdge;
                if (j + q < rows) u[q] = S[(size_t)(j + q) * kWave];
            }
        };
        uint32_t i = 0, j = 0, u[U], nu[U];
        uint32_t v = first * kWave + ln, nv = v, din = degree(v), ndin = din;
        auto own = pre(v < n, v), nown = own;
        load(0, 0, u);
        CSum s{0.f, 0.f};
        while (i < cnt) {
            if (j == 0 && i + 1 < cnt) {
                nv = v + nwaves * kWave;
                ndin = degree(nv);
                nown = pre(nv < n, nv);
            }
            const uint32_t rows = lane_value(nrow, (int)i);
            const bool last = j + U >= rows;
            const uint32_t ni = last ? i + 1 : i, nj = last ? 0u : j + U;
            if (ni < cnt) load(ni, nj, nu);
            if (rows) {
                float cv[U];
                gather.get(u, cv);
#pragma unroll
                for (uint32_t q = 0; q < U; q++) csum_add(s, cv[q]);
            }
            if (last) {
                done(din <= kPullHubDegree, v, own, s);
                s = CSum{0.f, 0.f};
                v = nv;
                din = ndin;
                own = nown;
            }
#pragma unroll
            for (uint32_t q = 0; q < U; q++) u[q] = nu[q];
            i = ni;
            j = nj;
        }
    }
}

// In-hubs of several chunks, once wait() has seen every block's chunk sums:
// eight lanes each (those of more than kHubWave chunks: the whole wave), dealt
// out so that the largest, which come first, fall to different waves; the
// first ones' data is loaded before the wait. done(has, v, own, sum),
// wave-convergent. Returns wait()'s result.
template <typename Wait, typename Pre, typename Done>
__device__ __forceinline__ bool wide_hub_sums(const DevGraph &g, const CSum *hubpart, const Bounds &bounds, uint32_t gwave,
                                              uint32_t nwaves, Wait wait, Pre pre, Done done)
{
    constexpr uint32_t kHubLanes = Bounds::kHubLanes, kHubs = kWave / kHubLanes, kHubWave = 8 * kHubLanes;
    const int ln = lane();
    Bounds bd = bounds;
    uint32_t h0 = gwave;
    auto own = pre(bd.chunks > 1, bd.v);
    if (!wait()) return false;
    while (h0 < g.nhubin) {
        const uint32_t cat = bd.at, cc = bd.chunks, cv = bd.v;
        const auto cown = own;
        h0 += nwaves * kHubs;
        if (h0 < g.nhubin) {
            bd.hub(g, h0, nwaves);
            own = pre(bd.chunks > 1, bd.v);
        }
        CSum s{0.f, 0.f};
        if (cc > 1 && cc <= kHubWave) {
#pragma unroll 8
            for (uint32_t k = (uint32_t)ln % kHubLanes; k < cc; k += kHubLanes) s = csum_merge(s, hubpart[cat + k]);
        }
        const CSum none{0.f, 0.f};
        s = csum_merge(s, dpp<kDppQuad1>(none, s));
        s = csum_merge(s, dpp<kDppQuad2>(none, s));
        s = csum_merge(s, dpp<kDppHalfMirror>(none, s));
        uint64_t wide = ballot(cc > kHubWave);
        while (wide) {
            const int l = first_lane(wide);
            const uint32_t wat = lane_value(cat, l), wc = lane_value(cc, l);
            CSum t{0.f, 0.f};
            for (uint32_t k = ln; k < wc; k += kWave) t = csum_merge(t, hubpart[wat + k]);
            t = wave_csum(t);
            if (ln / (int)kHubLanes == l / (int)kHubLanes) s = t;
            wide &= ~(0xFFull << l);
        }
        done(ln % (int)kHubLanes == 0 && cc > 1, cv, cown, s);
    }
    return true;
}

struct PrArgs {
    DevGraph g;
    float *x;          // ranks [n]
    float *contrib;    // 2 rows: x[u] / outdeg(u) of the current / next iteration
    CSum *hubpart;     // [nhugein] chunk sums
    PrPart *part;      // 2 x kMaxBlocks (residual, dangling) partials
    GridBarrier bar;
    uint32_t *abort;
    DevStats *stats;
    DevTrace *trace;
    double damping, tol;
    uint32_t max_iter;
    uint32_t probe;
};

// What bounds an iteration: the in-edges whose source has no place in LDS,
// each an L2 request for a line of which it needs 4 bytes. RMAT-21 (32.4 M
// edges, 36 % of them such), 17 iterations: 1778 us, of which 1030 are these
// reads (11.7 M an iteration at 0.19 T/s; the L2s answer 0.27 T/s at most),
// 210 the barriers, partial sums and LDS copy, the rest index reads, LDS reads
// and the vertices' own data. It took 2640 us when each in-edge's LDS or L2 read
// waited for the one before it, the chunks' bounds were read group by group,
// and every hub, also one of a single chunk, took a wave after the barrier.
template <int BS>
__global__ __launch_bounds__(BS) void k_pr_pull(PrArgs a)
{
    if (a.probe) {
        residency_probe(a.bar.words, 1u << 20);
        return;
    }
    constexpr int WPB = BS / kWave;
    const DevGraph &g = a.g;
    const uint32_t n = g.n, W = g.words;
    const uint32_t gtid = blockIdx.x * BS + threadIdx.x;
    const uint32_t nthreads = gridDim.x * BS;
    const uint32_t gwave = blockIdx.x * WPB + threadIdx.x / kWave;
    const uint32_t nwaves = gridDim.x * WPB;
    const int ln = lane();
    const uint32_t xcc = xcc_id();
    BarState gen = bar_begin(a.bar, xcc);
    const long long t_start = wall_clock64();
    const float df = (float)a.damping;
    const float inv_nf = (float)(1.0 / (double)n);
    const uint64_t stride = contrib_stride(n);

    __shared__ PrPart s_red[WPB];
    // as many ids in LDS as fit beside the rest: with 32 per thread RMAT-21
    // takes 1752 us, with 39 1708, 400 001 vertices 500 and 480
#ifndef SG_PR_LDS
#define SG_PR_LDS 39
#endif
    using Hot = Staged<BS, SG_PR_LDS>;
    __shared__ __align__(16) float s_cc[Hot::kLds + 4];

    // the block's (residual, dangling) partials, in a fixed order
    auto put_part = [&](uint32_t it, double res, CSum dang) {
        res = wave_sum_f64(res);
        dang = wave_csum(dang);
        if (ln == 0) s_red[threadIdx.x / kWave] = PrPart{res, dang.hi, dang.lo};
        __syncthreads();
        if (threadIdx.x < kWave) {
            const PrPart t = ln < WPB ? s_red[ln] : PrPart{0.0, 0.f, 0.f};
            res = wave_sum_f64(t.res);
            dang = wave_csum(CSum{t.dhi, t.dlo});
            if (ln == 0) a.part[(size_t)(it & 1) * kMaxBlocks + blockIdx.x] = PrPart{res, dang.hi, dang.lo};
        }
    };

    // x = 1/n; contributions of iteration 0; dangling mass
    CSum dang{0.f, 0.f};
    for (uint32_t v = gtid; v < n; v += nthreads) {
        a.x[v] = inv_nf;
        const uint32_t dout = g.row[v + 1] - g.row[v];
        a.contrib[v] = dout ? inv_nf / (float)dout : 0.0f;
        if (!dout) csum_add(dang, inv_nf);
    }
    if (threadIdx.x == 0) s_cc[Hot::kLds] = 0.f;
    put_part(0, 0.0, dang);
    bool ok = grid_sync(a.bar, xcc, gen, a.abort);

    const Bounds bounds(g, gwave, nwaves);
    uint32_t it = 0;
    double res = INFINITY;
    while (ok) {
        const float *cc = a.contrib + (size_t)(it & 1) * stride;
        float *cn = a.contrib + (size_t)((it + 1) & 1) * stride;
        // the LDS copy's loads are in flight while the partials are added
        Hot::take(s_cc, cc, n);
        // every wave adds the blocks' partials by itself: no wait for others
        double gres = 0.0;
        CSum gdang{0.f, 0.f};
        for (uint32_t i = ln; i < gridDim.x; i += kWave) {
            const PrPart q = a.part[(size_t)(it & 1) * kMaxBlocks + i];
            gres += q.res;
            gdang = csum_merge(gdang, CSum{q.dhi, q.dlo});
        }
        gres = wave_sum_f64(gres);
        gdang = wave_csum(gdang);
        if (it > 0) res = gres;
        if ((it > 0 && res < a.tol) || it >= a.max_iter) {
            Hot::wait();  // no copy into LDS outlives the block
            break;
        }
        const float base = (1.0f - df) * inv_nf + df * csum_value(gdang) * inv_nf;
        if (gtid == 0 && it < kTraceRows) {
            DevTrace t;
            t.round = it;
            t.variant = SG_SYNC_PULL_TD;
            t.in_nodes = n;
            t.pad = 0;
            t.in_edges = g.m;
            t.ticks = (unsigned long long)(wall_clock64() - t_start);
            a.trace[it] = t;
        }
        Hot::wait();
        __syncthreads();
        const Gather<Hot::kLds> gather{cc, s_cc, n};
        constexpr uint32_t kRows = 8;  // RMAT-21 1740 us by 4, 1708 by 8; 15 001 vertices 257 and 234
        double r_acc = 0.0;
        CSum d_acc{0.f, 0.f};
        struct Own {
            uint32_t dout;
            float xo;
        };
        auto pre = [&](bool has, uint32_t v) {
            return has ? Own{g.row[v + 1] - g.row[v], a.x[v]} : Own{0u, 0.f};
        };
        // x(v) from its in-edge sum, its last rank and its out-degree: FP32
        // ranks and contributions, the residual |x' - x| summed in FP64
        auto finish = [&](bool has, uint32_t v, const Own &o, const CSum &s) {
            if (!has) return;
            const float xn = base + df * csum_value(s);
            r_acc += fabs((double)xn - (double)o.xo);
            a.x[v] = xn;
            if (o.dout) cn[v] = xn / (float)o.dout;
            else csum_add(d_acc, xn);
        };
        // in-hubs of several chunks wait for every block's sums: arrive after
        // the chunks, wait once the other vertices are done
        hub_chunk_sums(g, gather, bounds, gwave, nwaves, pre,
                       [&](bool has, uint32_t c, uint32_t v, bool one, const Own &o, const CSum &s) {
                           if (has && !one) a.hubpart[c] = s;
                           finish(has && one, v, o, s);
                       });
        grid_signal(a.bar, xcc, gen, a.abort);
        word_sums<kRows>(g, gather, bounds, gwave, nwaves, pre, finish);
        ok = wide_hub_sums(g, a.hubpart, bounds, gwave, nwaves, [&]() { return grid_wait(a.bar, gen, a.abort); }, pre, finish);
        if (!ok) break;
        put_part(it + 1, r_acc, d_acc);
        it++;
        ok = grid_sync(a.bar, xcc, gen, a.abort);
    }

    if (gtid == 0) {
        DevStats s{};
        s.rounds = it;
        s.pull_rounds = it;
        s.iterations = it;
        s.residual = res;
        s.status = ok ? SG_OK : SG_ERR_TIMEOUT;
        *a.stats = s;
        if (it < kTraceRows) {
            DevTrace t{};
            t.round = it;
            t.variant = -1;
            t.ticks = (unsigned long long)(wall_clock64() - t_start);
            a.trace[it] = t;
        }
    }
    bar_end(a.bar);
}

// ------------------------------------------------------- residual DD kernel

struct PrDdArgs {
    DevGraph g;
    float *x;          // normalised ranks [n] (output)
    CSum *y;           // unnormalised ranks [n], compensated FP32
    float *r;          // residuals [n]: r + rlo, the rounding error of every
    float *rlo;        // atomic addition into r collected in rlo
    float *p;          // 2 rows: d r / outdeg of this / the next round's active vertices
    CSum *hubpart;     // [nhugein] chunk sums of pull rounds
    uint64_t *abit;    // 2 x W: active vertices of rounds k (k % 2)
    uint32_t *queue;   // 2 x qcap: vertices whose residual crossed theta
    uint32_t qcap;
    FrontierCtr *ctr;  // [0,1]: activation totals; [2,3,4]: queue appends
    PrPart *part;      // 2 x kMaxBlocks partials: pull rounds' counts, the final sums
    GridBarrier bar;
    uint32_t *abort;
    DevStats *stats;
    DevTrace *trace;
    double damping, theta, alpha;
    double total_wl;
    int32_t force;     // -1 auto, 0 push, 1 pull
    uint32_t max_rounds;
    uint32_t probe;
    int32_t it_force;    // ITERATIVE: -1, or the variant every round runs (kItPullTd...)
    float ticks_per_us;  // wall clock rate
    float cut;           // sample-based priority for ASYNC_PUSH_TD rounds (0: off)
};

// Sample-based priority (GetPriorityThreshold, include/framework/algo_variants.cuh:98-131;
// PRIORITY_SAMPLE_SIZE, graph_datum.cuh:18): a round's threshold is the
// residual at index size * (1 - cut) of size sampled residuals in ascending
// order, and only vertices at or above it push (IsHighPriority,
// samples/hybrid_pr/hybrid_pr.cu:117-121).
constexpr uint32_t kPrioSample = 1000;
constexpr uint32_t kPrioSort = 1024;  // sample padded to a power of two

__device__ __forceinline__ uint64_t sample_hash(uint64_t z)
{
    // SplitMix64 finaliser (Steele, Lea & Flood, OOPSLA 2014)
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// Every block draws the same vertices (a hash of round and index) and sorts
// their residuals in LDS (bitonic); residuals other blocks have already moved
// out this round read as 0, which can only lower a block's threshold.
template <int BS>
__device__ double sampled_threshold(const PrDdArgs &a, uint32_t k, double *s_smp)
{
    const uint32_t n = a.g.n, size = min(kPrioSample, n);
    for (uint32_t i = threadIdx.x; i < kPrioSort; i += BS)
        s_smp[i] = i < size ? (double)a.r[(uint32_t)(sample_hash(((uint64_t)k << 32) | i) % n)] : __builtin_inf();
    __syncthreads();
    for (uint32_t len = 2; len <= kPrioSort; len <<= 1) {
        for (uint32_t j = len >> 1; j > 0; j >>= 1) {
            for (uint32_t i = threadIdx.x; i < kPrioSort; i += BS) {
                const uint32_t p = i ^ j;
                if (p > i) {
                    const double x = s_smp[i], y = s_smp[p];
                    if ((x > y) == ((i & len) == 0)) {
                        s_smp[i] = y;
                        s_smp[p] = x;
                    }
                }
            }
            __syncthreads();
        }
    }
    const uint32_t at = min((uint32_t)((float)size * (1.0f - a.cut)), size - 1);
    const double t = s_smp[at];
    __syncthreads();
    return t;
}

// The ITERATIVE scheme's variant set in its std::set order
// (include/framework/hybrid_policy.h:172-186; AlgoVariant::operator< compares
// model, message passing, scheduling with SYNC < ASYNC, PUSH < PULL, TD < DD).
enum { kItPullTd = 0, kItPushTd = 1, kItPushDd = 2 };

// Replicated in every block: each computes the same decisions from the same
// barrier stamps and counters (PolicyDecisionMaker::GetNextPolicy and
// PredicateRunningTime, hybrid_policy.h:130-169,246-264; times are float as
// in its RunningInfo).
struct IterativePolicy {
    float time[3] = {0.f, 0.f, 0.f};  // last measured round time of each variant (us)
    float time_per_work = 0.f;
    float last_in_wl = 0.f;  // input workload (out-degree sum) of the last round
    int last = -1;

    // Record the round just finished (variant `v`, `us` long, `in_wl` input edges).
    __device__ void record(int v, float us, float in_wl)
    {
        time[v] = us;
        last = v;
        last_in_wl = in_wl;
    }

    // Variant for round k, `out_wl` = out-degree sum of the current worklist.
    __device__ int next(uint32_t k, float out_wl)
    {
        if (k < 3) return (int)k;  // inspection
        if (last == kItPushDd) time_per_work = time[kItPushDd] / last_in_wl;
        const float pred[3] = {time[kItPullTd], time[kItPushTd], time_per_work * out_wl};
        int best = 0;
        for (int v = 1; v < 3; v++)
            if (pred[v] < pred[best]) best = v;  // std::min_element: first minimum
        return best;
    }
};

// What the propagation of one residual round shares.
struct DdRound {
    const PrDdArgs *a;
    const float *p;    // this round's row
    double theta;
    Stager S;
    unsigned long long count;
    unsigned long long qscout;  // out-degree sum of queued vertices (ITERATIVE)
    bool qdeg;
};

// Add `add` to v's residual atomically, queueing v if this addition took its
// residual across theta. The addition returns the old value, so the lane
// recomputes the rounded sum it stored and adds its rounding error (TwoSum,
// Knuth) to rlo[v]. The crossing is told by r[v] alone, as stored before and
// after: additions only raise it, so one of them sees it cross, and a vertex that is
// left inactive is stored with its r below theta (csum_settle). Told by the
// exact sum, or with hi >= theta > hi + lo left in place, a residual could get
// past theta unseen and grow to the end of the run. Wave-convergent.
__device__ __forceinline__ void dd_accumulate(DdRound &R, bool act, uint32_t v, float add)
{
    bool crossed = false;
    if (act && add > 0.f) {
        const float old = atomicAdd(&R.a->r[v], add);
        const float s = old + add;
        const float bb = s - old;
        const float err = (old - (s - bb)) + (add - bb);
        if (err != 0.f) atomicAdd(&R.a->rlo[v], err);
        crossed = (double)old < R.theta && (double)s >= R.theta;
        R.count += crossed;
        if (crossed && R.qdeg) R.qscout += R.a->g.row[v + 1] - R.a->g.row[v];
    }
    stage(R.S, crossed, v);
}

// Push the active vertices of one word (one lane per vertex): wave-level
// prefix-sum scheduling of their out-edges; hubs go through the chunk list.
__device__ __forceinline__ void dd_push_word(DdRound &R, uint64_t word, uint32_t w)
{
    const PrDdArgs &a = *R.a;
    const DevGraph &g = a.g;
    const int ln = lane();
    const uint32_t u = w * 64 + ln;
    uint32_t b = 0, dg = 0;
    float pu = 0.f;
    if ((word >> ln) & 1) {
        b = g.row[u];
        dg = g.row[u + 1] - b;
        if (dg > kHugeDegree) dg = 0;
        if (dg) pu = R.p[u];
    }
    const uint32_t incl = wave_incl_scan(dg);
    const uint32_t total = lane_value(incl, kWave - 1);
    const uint32_t off = b - (incl - dg);
    for (uint32_t jb = 0; jb < total; jb += kWave) {
        const uint32_t j = jb + ln;
        const bool act = j < total;
        const int k = owner_lane(incl, j);
        const uint32_t e = shfl(off, k) + j;
        const float pk = __shfl(pu, k, kWave);
        const uint32_t v = act ? g.col[e] : 0u;
        dd_accumulate(R, act, v, pk);
    }
}

// kIter: rounds chosen by the ITERATIVE scheme's predicted times. Its state is
// not kept by the other runs' kernel, which has few registers to spare.
template <int BS, bool kIter>
__global__ __launch_bounds__(BS) void k_pr_dd(PrDdArgs a)
{
    if (a.probe) {
        residency_probe(a.bar.words, 1u << 20);
        return;
    }
    constexpr int WPB = BS / kWave;
    constexpr uint32_t kLdsQ = 4u * BS;
    const DevGraph &g = a.g;
    const uint32_t n = g.n, W = g.words;
    const uint32_t gtid = blockIdx.x * BS + threadIdx.x;
    const uint32_t nthreads = gridDim.x * BS;
    const uint32_t gwave = blockIdx.x * WPB + threadIdx.x / kWave;
    const uint32_t nwaves = gridDim.x * WPB;
    const int ln = lane();
    const uint32_t xcc = xcc_id();
    BarState gen = bar_begin(a.bar, xcc);
    const long long t_start = wall_clock64();
    const double d = a.damping, theta = a.theta;
    FrontierCtr *act_ctr = a.ctr;       // 2 slots
    FrontierCtr *q_ctr = a.ctr + 2;     // 3 slots

    __shared__ double s_smp[kIter ? kPrioSort : 1];
#ifndef SG_PRDD_LDS
#define SG_PRDD_LDS 30
#endif
    using Hot = Staged<BS, SG_PRDD_LDS>;
    __shared__ __align__(16) float s_p[Hot::kLds + 4];
    if (threadIdx.x == 0) s_p[Hot::kLds] = 0.f;
    __shared__ PrPart s_red2[WPB];
    __shared__ PrPart s_glob;
    __shared__ unsigned long long s_red[2][WPB];
    __shared__ unsigned long long s_lvl[5];
    __shared__ uint32_t s_q[kLdsQ];
    __shared__ uint32_t s_qn, s_flush[2];

    const float r0 = (float)((1.0 - d) / (double)n);
    const float df = (float)d;
    for (uint32_t v = gtid; v < n; v += nthreads) {
        a.y[v] = CSum{0.f, 0.f};
        a.r[v] = r0;
        a.rlo[v] = 0.f;
    }
    for (uint32_t w = gtid; w < 2 * W; w += nthreads) a.abit[w] = 0;
    if (blockIdx.x == 0) {
        for (int s = 0; s < 5; s++) clear_ctr(&a.ctr[s]);
    }
    // stamped barriers: the block completing each one records the wall clock,
    // so every block derives the same round times for the ITERATIVE scheme
    bool ok = grid_sync<kIter>(a.bar, xcc, gen, a.abort);
    __shared__ unsigned long long s_stamp;
    IterativePolicy ipol;
    unsigned long long stamp0 = 0, stamp_prev = 0;
    float in_wl_prev = 0.f;
    int v_prev = -1;
    bool held = false;  // the last activation held residuals >= theta back (priority)

    uint32_t k = 0, pushes = 0, pulls = 0;
    unsigned long long ptrace = 0;
    float *pc = a.p, *pn = a.p + contrib_stride(n);  // this round's and the next round's row of p
    while (ok) {
        if (a.max_rounds && k >= a.max_rounds) break;
        // ---- activation: move residual >= theta into y, set p and the bit
        if (kIter && threadIdx.x == 0) s_stamp = barrier_stamp(a.bar);
        read_counts(&q_ctr[k % 3], s_lvl);
        __syncthreads();
        const RoundCounts qc = unpack_counts(s_lvl, a.qcap);
        const unsigned long long stamp = s_stamp;
        __syncthreads();
        // ITERATIVE: time the round that just ended, then pick this round's
        // variant (topology-driven ones rebuild the active set by a scan)
        int var = -1;
        if (kIter) {
            if (k == 0) {
                stamp0 = stamp;
            } else {
                const float us = (float)((double)(stamp - stamp_prev) / (double)a.ticks_per_us);
                ipol.record(v_prev, us, in_wl_prev);
                if (gtid == 0 && k - 1 < kTraceRows) a.trace[k - 1].ticks = stamp - stamp0;
            }
            stamp_prev = stamp;
            var = a.it_force >= 0 ? a.it_force : ipol.next(k, (float)qc.scout);
        }
        uint64_t *ab = a.abit + (size_t)(k & 1) * W;
        unsigned long long scout = 0, cnt = 0;
        auto activate = [&](uint32_t u, float ru) {
            CSum yu = a.y[u];
            csum_add(yu, ru);
            a.y[u] = yu;
            const uint32_t dout = g.row[u + 1] - g.row[u];
            if (dout) pc[u] = df * ru / (float)dout;
            scout += dout;
            cnt++;
        };
        bool waiting = false;  // this lane saw a residual >= theta left below the priority threshold
        // a scan also after a round that held residuals back: they did not
        // cross theta again, so no queue holds them
        // or once the queue holds an eighth of the vertices (it holds every
        // residual >= theta, so a scan finds the same set): reading all residuals
        // in order then costs less than two returning atomics per entry
        const bool scan = k == 0 || qc.overflow || held || var == kItPullTd || var == kItPushTd || qc.qlen > n / 8;
        if (scan) {
            double thr = theta;
            if (kIter && var == kItPushTd && a.cut > 0.f) thr = fmax(theta, sampled_threshold<BS>(a, k, s_smp));
            for (uint32_t w = gwave; w < W; w += nwaves) {
                const uint32_t v = w * 64 + ln;
                bool act = false;
                if (v < n) {
                    const CSum c{a.r[v], a.rlo[v]};
                    const float rv = csum_value(c);
                    act = (double)rv >= thr;
                    waiting |= !act && (double)rv >= theta;
                    if (act) {
                        a.r[v] = 0.f;
                        a.rlo[v] = 0.f;
                        activate(v, rv);
                    } else {
                        pc[v] = 0.f;  // a pull round reads every source's
                        if ((double)rv < theta && (double)c.hi >= theta) {
                            const CSum s = csum_settle(c);
                            a.r[v] = s.hi;
                            a.rlo[v] = s.lo;
                        }
                    }
                }
                const uint64_t m = ballot(act);
                if (ln == 0) ab[w] = m;
            }
        } else {
            const uint32_t *qin = a.queue + (size_t)(k & 1) * a.qcap;
            for (uint32_t i = gtid; i < qc.qlen; i += nthreads) {
                const uint32_t u = qin[i];
                // claim the residual: a vertex queued twice is activated once
                // (no propagation runs in this phase; a claim split between
                // two copies returns the part it took)
                const float hi = atomicExch(&a.r[u], 0.f);
                const float lo = atomicExch(&a.rlo[u], 0.f);
                const float ru = hi + lo;
                if ((double)ru >= theta) {
                    atomicOr((unsigned long long *)&ab[u >> 6], 1ull << (u & 63));
                    activate(u, ru);
                } else if (hi != 0.f || lo != 0.f) {
                    const CSum c = hi != 0.f ? csum_settle(CSum{hi, lo}) : CSum{0.f, lo};
                    atomicAdd(&a.r[u], c.hi);
                    atomicAdd(&a.rlo[u], c.lo);
                }
            }
        }
        // the slot's has_huge flag carries "residuals >= theta were held back"
        publish_counts<WPB>(&act_ctr[k & 1], scout, cnt, waiting, s_red);
        ok = grid_sync(a.bar, xcc, gen, a.abort);
        if (!ok) break;

        // ---- propagation
        read_counts(&act_ctr[k & 1], s_lvl);
        if (threadIdx.x == 0) s_qn = 0;
        __syncthreads();
        const RoundCounts ac = unpack_counts(s_lvl, a.qcap);
        __syncthreads();
        if (ac.count == 0 && !ac.has_huge) break;  // every residual is below theta
        held = ac.has_huge;
        auto pulls_at = [&](unsigned long long sc) {
            return a.force >= 0 ? a.force == 1 : (double)sc > a.total_wl / a.alpha;
        };
        bool pull;
        if (var >= 0) pull = var == kItPullTd;
        else pull = pulls_at(ac.scout);
        auto note_round = [&](bool was_pull, const RoundCounts &c) {
            if (was_pull) {
                pulls++;
                if (k < 64) ptrace |= 1ull << k;
            } else {
                pushes++;
            }
            if (var < 0 && gtid == 0) write_trace(a.trace, k, was_pull, c.count, c.scout, t_start);
        };
        note_round(pull, ac);
        if (var >= 0) {
            // the reference's input workload: edges for a topology-driven
            // round, the worklist's out-degree sum for a data-driven one
            in_wl_prev = var == kItPushDd ? (float)ac.scout : (float)g.m;
            v_prev = var;
            if (gtid == 0 && k < kTraceRows) {
                DevTrace t{};
                t.round = k;
                t.variant = var == kItPullTd ? SG_SYNC_PULL_TD : var == kItPushTd ? SG_ASYNC_PUSH_TD : SG_ASYNC_PUSH_DD;
                t.in_nodes = (uint32_t)ac.count;
                t.in_edges = ac.scout;
                a.trace[k] = t;  // ticks filled in when the round's end is known
            }
        }
        DdRound R;
        R.a = &a;
        R.theta = theta;
        R.qdeg = kIter;
        // counters and bitmap of the rounds to come, and the queue of the next
        auto begin_round = [&]() {
            if (blockIdx.x == 0) {
                clear_ctr(&act_ctr[(k + 1) & 1]);
                clear_ctr(&q_ctr[(k + 2) % 3]);
            }
            R.p = pc;
            R.S = Stager{a.queue + (size_t)((k + 1) & 1) * a.qcap, a.qcap, &q_ctr[(k + 1) % 3], s_q, &s_qn, kLdsQ};
            R.count = 0;
            R.qscout = 0;
        };
        begin_round();
        if (pull && !scan) {
            // the round's row of p still holds earlier rounds' entries
            for (uint32_t v = gtid; v < n; v += nthreads)
                if (!test_bit(ab, v)) pc[v] = 0.f;
            ok = grid_sync(a.bar, xcc, gen, a.abort);
            if (!ok) break;
        }
        // ---- pull rounds: each vertex adds what its in-edges bring and, if
        // that takes its residual to theta, is activated for the next round in
        // the same pass (the next row of p), with no queue and no pass over the
        // residuals in between: a round of two grid barriers and one reading of
        // the edges, as one of the power iteration. Rounds of the ITERATIVE
        // scheme, and the last one before max_rounds, leave activation out.
        // RMAT graph of 100 003 vertices, 1.4 M edges, nearly all active: 21 us a
        // round, 2.2 ms a run (45 and 4.8 with activation in a pass of its own);
        // ~10 of them are the two barriers, the counts and the LDS copy, the rest the
        // words' chains of in-edge steps and the hubs.
        bool more = true;
        const Bounds bounds(g, gwave, nwaves);
        if (pull) Hot::take(s_p, pc, n);
        while (pull) {
            const bool act_next = !kIter && !(a.max_rounds && k + 1 >= a.max_rounds);
            Hot::wait();
            __syncthreads();
            const Gather<Hot::kLds> gather{pc, s_p, n};
            constexpr uint32_t kRows = BS > 512 ? 8 : 16;  // 100 003 vertices, 512 threads: 2356 us by 8, 2255 by 16
            unsigned long long nscout = 0, ncnt = 0;
            struct Own {
                uint32_t dout;
                CSum r;
            };
            struct Later {};  // loaded at the end
            auto pre = [&](bool has, uint32_t v) {
                Own o{0u, CSum{0.f, 0.f}};
                if (has) {
                    o.dout = g.row[v + 1] - g.row[v];
                    o.r = CSum{a.r[v], a.rlo[v]};
                }
                return o;
            };
            auto finish = [&](bool has, uint32_t v, const Own &o, const CSum &add) {
                CSum c = csum_merge(o.r, add);
                const float ru = csum_value(c);
                const bool active = has && act_next && (double)ru >= theta;
                bool crossed = false;
                if (has && act_next) {
                    float pv = 0.f;
                    if (active) {
                        CSum yv = a.y[v];
                        csum_add(yv, ru);
                        a.y[v] = yv;
                        if (o.dout) pv = df * ru / (float)o.dout;
                        nscout += o.dout;
                        ncnt++;
                        c = CSum{0.f, 0.f};
                    }
                    pn[v] = pv;
                }
                if (has && (csum_value(add) > 0.f || active)) {
                    if (!active) c = csum_settle(c);
                    a.r[v] = c.hi;
                    a.rlo[v] = c.lo;
                    crossed = kIter && (double)o.r.hi < theta && (double)c.hi >= theta;
                    R.count += crossed;
                    if (crossed && R.qdeg) R.qscout += o.dout;
                }
                if (kIter) stage(R.S, crossed, v);
            };
            auto later = [](bool, uint32_t) { return Later{}; };
            hub_chunk_sums(g, gather, bounds, gwave, nwaves, later,
                           [&](bool has, uint32_t c, uint32_t v, bool one, Later, const CSum &s) {
                               if (has && !one) a.hubpart[c] = s;
                               finish(has && one, v, pre(has && one, v), s);
                           });
            grid_signal(a.bar, xcc, gen, a.abort);
            word_sums<kRows>(g, gather, bounds, gwave, nwaves, pre, finish);
            ok = wide_hub_sums(
                g, a.hubpart, bounds, gwave, nwaves, [&]() { return grid_wait(a.bar, gen, a.abort); }, later,
                [&](bool has, uint32_t v, Later, const CSum &s) { finish(has, v, pre(has, v), s); });
            if (!ok || !act_next) break;
            // the next round's totals, by blocks: no atomics, and every wave
            // adds them by itself
            nscout = wave_sum_u64(nscout);
            ncnt = wave_sum_u64(ncnt);
            if (ln == 0) {
                s_red[0][threadIdx.x / kWave] = nscout;
                s_red[1][threadIdx.x / kWave] = ncnt;
            }
            __syncthreads();
            if (threadIdx.x < kWave) {
                nscout = wave_sum_u64(ln < WPB ? s_red[0][ln] : 0ull);
                ncnt = wave_sum_u64(ln < WPB ? s_red[1][ln] : 0ull);
                if (ln == 0)
                    ((ulonglong2 *)a.part)[(size_t)((k + 1) & 1) * kMaxBlocks + blockIdx.x] = make_ulonglong2(nscout, ncnt);
            }
            ok = grid_sync(a.bar, xcc, gen, a.abort);
            if (!ok) break;
            k++;
            {
                float *const t = pc;
                pc = pn;
                pn = t;
            }
            Hot::take(s_p, pc, n);  // in flight while the counts are added
            RoundCounts nc{};
            for (uint32_t i = ln; i < gridDim.x; i += kWave) {
                const ulonglong2 q = ((const ulonglong2 *)a.part)[(size_t)(k & 1) * kMaxBlocks + i];
                nc.scout += q.x;
                nc.count += q.y;
            }
            nc.scout = wave_sum_u64(nc.scout);
            nc.count = wave_sum_u64(nc.count);
            if (nc.count == 0) {
                more = false;  // every residual is below theta
                Hot::wait();   // no copy into LDS outlives the block
                break;
            }
            pull = pulls_at(nc.scout);
            note_round(pull, nc);
            if (!pull) {
                // a push round reads the active set off its bitmap, and finds
                // clear counters
                if (blockIdx.x == 0) {
                    for (int c = 0; c < 5; c++) clear_ctr(&a.ctr[c]);
                }
                ab = a.abit + (size_t)(k & 1) * W;
                begin_round();
                for (uint32_t w = gwave; w < W; w += nwaves) {
                    const uint32_t v = w * 64 + ln;
                    const uint64_t m = ballot(v < n && pc[v] != 0.f);
                    if (ln == 0) ab[w] = m;
                }
                ok = grid_sync(a.bar, xcc, gen, a.abort);
            }
        }
        if (!ok || !more) break;
        uint64_t *ab_next = a.abit + (size_t)((k + 1) & 1) * W;
        for (uint32_t w = gtid; w < W; w += nthreads) ab_next[w] = 0;
        if (!pull) {
            for (uint32_t c0 = 0; c0 < g.nhuge; c0 += nwaves * kWave) {
                const uint32_t c = c0 + (uint32_t)ln * nwaves + gwave;
                uint2 dsc = make_uint2(0u, 0u);
                bool mem = false;
                if (c < g.nhuge) {
                    dsc = g.huge[c];
                    mem = test_bit(ab, dsc.x);
                }
                uint64_t mm = ballot(mem);
                while (mm) {
                    const int t = first_lane(mm);
                    mm &= mm - 1;
                    const uint32_t u = lane_value(dsc.x, t), beg = lane_value(dsc.y, t);
                    const uint32_t end = min(g.row[u + 1], beg + kHugeChunk);
                    const float pu = pc[u];
                    for (uint32_t e0 = beg; e0 < end; e0 += kWave) {
                        const uint32_t e = e0 + ln;
                        const bool act = e < end;
                        dd_accumulate(R, act, act ? g.col[e] : 0u, pu);
                    }
                }
            }
            for (uint32_t w = gwave; w < W; w += nwaves) {
                const uint64_t word = ab[w];
                if (word) dd_push_word(R, word, w);
            }
        }
        publish_counts<WPB>(&q_ctr[(k + 1) % 3], R.qscout, R.count, false, s_red);
        flush_stage(R.S, s_flush);
        k++;
        ok = grid_sync<kIter>(a.bar, xcc, gen, a.abort);
    }

    // ---- absorb what residual is left, then normalise
    // the sum of y (compensated FP32) normalises; the residual mass absorbed
    // here is reduced in FP64
    CSum ysum{0.f, 0.f};
    double rsum = 0.0;
    if (ok) {
        for (uint32_t v = gtid; v < n; v += nthreads) {
            CSum yv = a.y[v];
            const float rv = a.r[v], rl = a.rlo[v];
            csum_add(yv, rv);
            csum_add(yv, rl);
            a.y[v] = yv;
            csum_add(ysum, csum_value(yv));
            rsum += (double)rv + (double)rl;
        }
        const PrPart t = block_part<WPB>(rsum, ysum, s_red2);
        // (the set that no block reads any more)
        if (threadIdx.x == 0) a.part[(size_t)((k + 1) & 1) * kMaxBlocks + blockIdx.x] = t;
        ok = grid_sync(a.bar, xcc, gen, a.abort);
    }
    PrPart tot{0.0, 1.f, 0.f};
    if (ok) {
        tot = grid_part<BS>(a.part + (size_t)((k + 1) & 1) * kMaxBlocks, gridDim.x, s_red2, &s_glob);
        const float ys = csum_value(CSum{tot.dhi, tot.dlo});
        const float inv = ys > 0.f ? 1.0f / ys : 0.f;
        for (uint32_t v = gtid; v < n; v += nthreads) a.x[v] = csum_value(a.y[v]) * inv;
    }
    if (gtid == 0) {
        DevStats s{};
        s.rounds = k;
        s.push_rounds = pushes;
        s.pull_rounds = pulls;
        s.trace = ptrace;
        s.iterations = k;
        s.residual = tot.res;  // residual mass absorbed at the end (unnormalised)
        s.status = ok ? SG_OK : SG_ERR_TIMEOUT;
        *a.stats = s;
        if (k < kTraceRows) {
            DevTrace t{};
            t.round = k;
            t.variant = -1;
            t.ticks = (unsigned long long)(wall_clock64() - t_start);
            a.trace[k] = t;
        }
    }
    bar_end(a.bar);
}

template <typename Args, void (*K)(Args)>
int launch_persistent(sg_engine *e, Args &args, int bs)
{
    sg_engine::PGrid *pg = nullptr;
    auto probe = [e, args, bs](int blocks, uint32_t *words) -> int {
        Args p = args;
        p.probe = 1;
        p.bar.words = words;
        void *params[] = {&p};
        SG_HIP(hipLaunchKernel((const void *)K, dim3(blocks), dim3(bs), params, 0, e->stream));
        return SG_OK;
    };
    int rc = engine_persistent_grid(e, (const void *)K, bs, probe, &pg);
    if (rc) return rc;
    if (pg->blocks > (int)kMaxBlocks) SG_FAIL(SG_ERR_STATE, "sg_pagerank: grid exceeds the partial-sum area");
    bind_barrier(pg, args.bar);
    return engine_launch_persistent(e, [&]() -> int {
        void *params[] = {&args};
        SG_HIP(hipLaunchKernel((const void *)K, dim3(pg->blocks), dim3(bs), params, 0, e->stream));
        pg->launches++;
        return SG_OK;
    });
}

}  // namespace

extern "C" int sg_pagerank(sg_engine *e, double damping, double tol, int32_t max_iter, int32_t mode)
{
    if (!e) SG_FAIL(SG_ERR_INVALID, "sg_pagerank: null engine");
    if (!(damping >= 0.0 && damping < 1.0)) SG_FAIL(SG_ERR_RANGE, "sg_pagerank: damping must be in [0, 1)");
    if (!(tol > 0.0)) SG_FAIL(SG_ERR_RANGE, "sg_pagerank: tol must be > 0");
    if (max_iter < 0) SG_FAIL(SG_ERR_RANGE, "sg_pagerank: max_iter < 0");
    const sg_engine_options &o = e->opt;
    if (o.lb_push == SG_LB_NONE || o.lb_pull == SG_LB_NONE)
        SG_FAIL(SG_ERR_UNSUPPORTED, "sg_pagerank: LoadBalancing::NONE applies to sg_bfs and sg_sssp only");
    if (mode == SG_PR_AUTO) {
        const int fv = o.force_variant;
        mode = (fv == SG_ASYNC_PUSH_DD || fv == SG_ASYNC_PULL_DD || fv == SG_SYNC_PUSH_DD || fv == SG_SYNC_PULL_DD)
                   ? SG_PR_PUSH_DD
                   : SG_PR_PULL_TD;
    }
    if (mode != SG_PR_PULL_TD && mode != SG_PR_PUSH_DD && mode != SG_PR_ITERATIVE)
        SG_FAIL(SG_ERR_INVALID, "sg_pagerank: unknown mode");
    int32_t it_force = -1;
    if (mode == SG_PR_ITERATIVE) {
        switch (o.force_variant) {
        case SG_VARIANT_AUTO: break;
        case SG_SYNC_PULL_TD: it_force = kItPullTd; break;
        case SG_ASYNC_PUSH_TD: it_force = kItPushTd; break;
        case SG_ASYNC_PUSH_DD: it_force = kItPushDd; break;
        default:
            SG_FAIL(SG_ERR_UNSUPPORTED,
                    "sg_pagerank: the ITERATIVE scheme runs SYNC_PULL_TD, ASYNC_PUSH_TD or ASYNC_PUSH_DD only");
        }
    }
    const DevGraph &d = e->g->dev;
    int rc = engine_ensure_bfs_state(e);
    if (rc) return rc;
    void *res = nullptr;
    if ((rc = engine_result_rows(e, 1, &res))) return rc;
    const uint64_t n = d.n;
    const int bs = o.block_size ? o.block_size : 1024;
    if (bs != 256 && bs != 512 && bs != 1024) SG_FAIL(SG_ERR_UNSUPPORTED, "sg_pagerank: block_size must be 256, 512 or 1024");
    e->last_algo = 2;
    const uint64_t part_bytes = 2ull * kMaxBlocks * sizeof(double2);
    if (mode == SG_PR_PULL_TD) {
        // contrib (two rows, 16-byte aligned) | hubpart | partials
        const uint64_t off_hub = 2ull * contrib_stride(d.n) * 4;
        const uint64_t off_part = off_hub + ((uint64_t)d.nhugein * 8 + 15) / 16 * 16;
        if ((rc = engine_ensure_aux(e, off_part + part_bytes))) return rc;
        char *base = (char *)e->aux;
        PrArgs a{};
        a.g = d;
        a.x = (float *)res;
        a.contrib = (float *)base;
        a.hubpart = (CSum *)(base + off_hub);
        a.part = (PrPart *)(base + off_part);
        a.bar.spin_limit = 1u << 22;
        a.abort = e->abort_flag;
        a.stats = e->stats;
        a.trace = e->trace;
        a.damping = damping;
        a.tol = tol;
        a.max_iter = max_iter ? (uint32_t)max_iter : 1000u;
        switch (bs) {
        case 256: rc = launch_persistent<PrArgs, k_pr_pull<256>>(e, a, 256); break;
        case 512: rc = launch_persistent<PrArgs, k_pr_pull<512>>(e, a, 512); break;
        default: rc = launch_persistent<PrArgs, k_pr_pull<1024>>(e, a, 1024); break;
        }
    } else {
        const int force = mode == SG_PR_ITERATIVE ? -1 : forced_direction(o);
        if (force < -1) SG_FAIL(SG_ERR_UNSUPPORTED, "sg_pagerank: data-driven mode takes push/pull DD variants only");
        // y (n compensated floats) | r | rlo (n floats each) | two rows of p | hubpart | partials
        const uint64_t off_hub = n * 16 + 2ull * contrib_stride(d.n) * 4;
        const uint64_t off_part = off_hub + ((uint64_t)d.nhugein * 8 + 15) / 16 * 16;
        if ((rc = engine_ensure_aux(e, off_part + part_bytes))) return rc;
        char *base = (char *)e->aux;
        PrDdArgs a{};
        a.g = d;
        a.x = (float *)res;
        a.y = (CSum *)base;
        a.r = (float *)(base + n * 8);
        a.rlo = (float *)(base + n * 12);
        a.p = (float *)(base + n * 16);
        a.hubpart = (CSum *)(base + off_hub);
        a.part = (PrPart *)(base + off_part);
        a.abit = e->bitmaps;
        a.queue = e->queues;
        a.qcap = e->qcap;
        a.ctr = (FrontierCtr *)e->ctr;
        a.bar.spin_limit = 1u << 22;
        a.abort = e->abort_flag;
        a.stats = e->stats;
        a.trace = e->trace;
        a.damping = damping;
        a.theta = tol * (1.0 - damping) / (double)n;
        a.alpha = o.alpha == 0.0 ? 1.0 : o.alpha;
        a.total_wl = (double)d.m * o.edge_factor;
        a.force = force;
        a.max_rounds = max_iter ? (uint32_t)max_iter : 100000u;
        const bool it = mode == SG_PR_ITERATIVE;
        a.it_force = it_force;
        a.ticks_per_us = (float)(e->wall_khz / 1000.0);
        a.cut = 0.f;
        if (mode == SG_PR_ITERATIVE && o.priority == SG_PRIO_SAMPLING) {
            if (!(o.cut_threshold > 0.f && o.cut_threshold < 1.f))
                SG_FAIL(SG_ERR_RANGE, "sg_pagerank: sample-based priority needs 0 < cut_threshold < 1");
            a.cut = o.cut_threshold;
        }
        // Up to 2^18 vertices a round is latency: blocks of 512 threads, whose
        // waves have registers for 16 rows in flight and none to spill (100 003
        // vertices 2255 us, of 1024 threads 2564; 400 001: 3768 and 3777). Beyond,
        // twice the waves hide more (1 000 001: 7340 and 6896).
        const int dbs = o.block_size || d.n > (1u << 18) ? bs : 512;
        switch (dbs) {
        case 256:
            rc = it ? launch_persistent<PrDdArgs, k_pr_dd<256, true>>(e, a, 256) : launch_persistent<PrDdArgs, k_pr_dd<256, false>>(e, a, 256);
            break;
        case 512:
            rc = it ? launch_persistent<PrDdArgs, k_pr_dd<512, true>>(e, a, 512) : launch_persistent<PrDdArgs, k_pr_dd<512, false>>(e, a, 512);
            break;
        default:
            rc = it ? launch_persistent<PrDdArgs, k_pr_dd<1024, true>>(e, a, 1024) : launch_persistent<PrDdArgs, k_pr_dd<1024, false>>(e, a, 1024);
        }
    }
    if (rc) return rc;
    if ((rc = engine_finish(e, 1))) return rc;
    e->timed = true;
    e->clocked = e->last_grid;
    return SG_OK;
}
