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
// stored as FP32. In the pull mode every sum (in-edges, dangling mass, L1
// residual) is FP64, in a fixed order for a given grid, so repeated runs give
// identical bits. In the residual mode the unnormalised ranks, the residuals
// (each atomic addition's rounding error, recomputed by the adding lane, goes
// to a second FP32 array) and the normalising sum are compensated FP32 (hi +
// lo, Neumaier); the residual mass absorbed at the end is reduced in FP64.
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
// from active sources when it exceeds m / alpha (pull).
#include "frontier.hpp"

using namespace sg;

namespace {

// ------------------------------------------------------------------ helpers

// ------------------------------------------- compensated FP32 accumulation
// A sum kept as hi + lo, where lo collects the rounding error of every
// addition into hi (Neumaier's variant of Kahan summation): FP32 storage and
// arithmetic with an error close to one rounding of the final sum.
struct CSum {
    float hi, lo;
};

__device__ __forceinline__ void csum_add(CSum &a, float x)
{
    const float s = a.hi + x;
    const float t = fabsf(a.hi) >= fabsf(x) ? (a.hi - s) + x : (x - s) + a.hi;
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

// Lanes of one row of 16 take each other's sums (every lane has the total).
__device__ __forceinline__ double row_sum(double x)
{
    x += dpp<kDppRowRor + 8>(0.0, x);
    x += dpp<kDppRowRor + 4>(0.0, x);
    x += dpp<kDppRowRor + 2>(0.0, x);
    x += dpp<kDppRowRor + 1>(0.0, x);
    return x;
}

// (FP64 adds run at the rate of FP32 ones here: a conversion and an add per
// in-edge where a compensated FP32 sum takes eight instructions.)
// Four wave sums together: lane l gets that of s[l % 4]. Halves of the wave,
// then rows of 16 lanes, trade places between two sums, so that three
// additions leave one sum per row, where four scans would take 24.
__device__ __forceinline__ double wave_sum4(const double (&s)[4])
{
    auto fold = [](double a, double b, bool half) {
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
        return a + b;
    };
    // rows of (0, 2): 0 0 2 2; of (1, 3): 1 1 3 3; of both: 0 1 2 3
    const double t = row_sum(fold(fold(s[0], s[2], true), fold(s[1], s[3], true), false));
    return shfl(t, (lane() & 3) * 16);
}

struct PrArgs {
    DevGraph g;
    float *x;          // ranks [n]
    float *contrib;    // 2 rows: x[u] / outdeg(u) of the current / next iteration
    double *hubpart;   // [nhugein] chunk sums
    double2 *part;     // 2 x kMaxBlocks (residual, dangling) partials
    GridBarrier bar;
    uint32_t *abort;
    DevStats *stats;
    DevTrace *trace;
    double damping, tol;
    uint32_t max_iter;
    uint32_t probe;
};

// Floats from one row of contributions to the next: 16-byte aligned rows.
__host__ __device__ constexpr uint64_t contrib_stride(uint32_t n) { return ((uint64_t)n + 3) / 4 * 4; }

// What bounds an iteration: the in-edges whose source has no place in LDS,
// each an L2 request for a line of which it needs 4 bytes. RMAT-21 (32.4 M
// edges, 36 % of them such), 17 iterations: 1800 us, of which 1030 are these
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
    constexpr uint32_t kPad = 0xFFFFFFFFu;  // no in-edge
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

    __shared__ double2 s_red[WPB];
    // The lowest ids' contributions (in a degree-ordered graph the sources of
    // most in-edges) are copied to LDS each iteration: they are read-only
    // until the next barrier, and the gather reads them there instead of
    // sending one L2 request per in-edge. As many as fit beside the rest: with
    // 32 per thread RMAT-21 takes 1848 us, with 39 1803.
#ifndef SG_PR_LDS
#define SG_PR_LDS 39
#endif
    constexpr uint32_t kCcLds = SG_PR_LDS * BS;
    __shared__ __align__(16) float s_cc[kCcLds + 4];  // [kCcLds]: 0, read for every other entry

    // the block's (residual, dangling) partials, in a fixed order
    auto put_part = [&](uint32_t it, double res, double dang) {
        res = wave_sum_f64(res);
        dang = wave_sum_f64(dang);
        if (ln == 0) s_red[threadIdx.x / kWave] = make_double2(res, dang);
        __syncthreads();
        if (threadIdx.x < kWave) {
            const double2 t = ln < WPB ? s_red[ln] : make_double2(0.0, 0.0);
            res = wave_sum_f64(t.x);
            dang = wave_sum_f64(t.y);
            if (ln == 0) a.part[(size_t)(it & 1) * kMaxBlocks + blockIdx.x] = make_double2(res, dang);
        }
    };

    // x = 1/n; contributions of iteration 0; dangling mass
    double dang = 0.0;
    for (uint32_t v = gtid; v < n; v += nthreads) {
        a.x[v] = inv_nf;
        const uint32_t dout = g.row[v + 1] - g.row[v];
        a.contrib[v] = dout ? inv_nf / (float)dout : 0.0f;
        if (!dout) dang += (double)inv_nf;
    }
    if (threadIdx.x == 0) s_cc[kCcLds] = 0.f;
    put_part(0, 0.0, dang);
    bool ok = grid_sync(a.bar, xcc, gen, a.abort);

    uint32_t it = 0;
    double res = INFINITY;
    while (ok) {
        const float *cc = a.contrib + (size_t)(it & 1) * stride;
        float *cn = a.contrib + (size_t)((it + 1) & 1) * stride;
        // the LDS copy's loads are in flight while the partials are added
        const uint32_t ncc = min(n, kCcLds);
        constexpr int kFill = (int)((kCcLds / 4 + BS - 1) / BS);
        float4 fill[kFill];
#pragma unroll
        for (int i = 0; i < kFill; i++) {
            fill[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (4 * threadIdx.x < ncc - min(ncc, (uint32_t)(4 * i * BS))) fill[i] = ((const float4 *)cc + i * BS)[threadIdx.x];
        }
        // every wave adds the blocks' partials by itself: no wait for others
        double2 gs = make_double2(0.0, 0.0);
        for (uint32_t i = ln; i < gridDim.x; i += kWave) {
            const double2 q = a.part[(size_t)(it & 1) * kMaxBlocks + i];
            gs.x += q.x;
            gs.y += q.y;
        }
        gs.x = wave_sum_f64(gs.x);
        gs.y = wave_sum_f64(gs.y);
        if (it > 0) res = gs.x;
        if ((it > 0 && res < a.tol) || it >= a.max_iter) break;
        const float base = (1.0f - df) * inv_nf + df * (float)gs.y * inv_nf;
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
#pragma unroll
        for (int i = 0; i < kFill; i++) {
            if (4 * threadIdx.x < ncc - min(ncc, (uint32_t)(4 * i * BS))) ((float4 *)s_cc + i * BS)[threadIdx.x] = fill[i];
        }
        __syncthreads();
        // contributions of N sources: the loads of those outside LDS are all
        // issued first, then every entry reads LDS (the zero, if it has no
        // place there), so no entry waits for the one before it
        const uint32_t ncold = n > kCcLds ? n - kCcLds : 0u;
        auto gather = [&](const uint32_t *u, float *c, auto N) {
#pragma unroll
            for (int q = 0; q < N.value; q++) {
                c[q] = 0.f;
                if (u[q] - kCcLds < ncold) c[q] = cc[u[q]];
            }
#pragma unroll
            for (int q = 0; q < N.value; q++) c[q] += s_cc[min(u[q], kCcLds)];
        };
        double r_acc = 0.0, d_acc = 0.0;
        // x(v) from its in-edge sum, its last rank and its out-degree: FP32
        // ranks and contributions, sums and the residual |x' - x| in FP64
        auto finish = [&](uint32_t v, double s, float xo, uint32_t dout) {
            const float xn = base + df * (float)s;
            r_acc += fabs((double)xn - (double)xo);
            a.x[v] = xn;
            if (dout) cn[v] = xn / (float)dout;
            else d_acc += (double)xn;
        };
        // (A1) chunk sums of the in-hubs, dealt out one by one. A lane holds
        // one chunk's bounds and, in the end, its sum; the wave adds kQ
        // chunks together, the next kQ chunks' in-edges in flight meanwhile.
        // A hub of one chunk is finished here.
        constexpr int kQ = 4, kSteps = (int)(kPullChunk / kWave);
        for (uint32_t first = gwave; first < g.nhugein; first += nwaves * kWave) {
            const uint32_t cnt = min((uint32_t)kWave, (g.nhugein - first + nwaves - 1) / nwaves);
            const uint32_t c = first + (uint32_t)ln * nwaves;
            uint32_t hv = 0, beg = 0, len = 0, dout = 0;
            float xo = 0.f;
            bool one = false;
            if ((uint32_t)ln < cnt) {
                const uint2 dsc = g.hugein[c];
                hv = dsc.x;
                beg = dsc.y;
                const uint32_t b = g.cstart[hv], e = g.cstart[hv + 1];
                len = min(e - beg, kPullChunk);
                one = e - b <= kPullChunk;
                dout = g.row[hv + 1] - g.row[hv];
                xo = a.x[hv];
            }
            auto load = [&](uint32_t j, uint32_t *u) {
#pragma unroll
                for (int q = 0; q < kQ; q++) {
                    const uint32_t l = lane_value(len, (int)j + q);
                    const uint32_t *src = g.csrc + lane_value(beg, (int)j + q);
#pragma unroll
                    for (int t = 0; t < kSteps; t++) {
                        const uint32_t k = (uint32_t)(t * kWave + ln);
                        u[q * kSteps + t] = k < l ? src[k] : kPad;
                    }
                }
            };
            double mine = 0.0;
            uint32_t u[kQ * kSteps], nu[kQ * kSteps];
            load(0, u);
            for (uint32_t j = 0; j < cnt; j += kQ) {
                if (j + kQ < cnt) load(j + kQ, nu);
                float cv[kQ * kSteps];
                gather(u, cv, std::integral_constant<int, kQ * kSteps>{});
                double s[kQ];
#pragma unroll
                for (int q = 0; q < kQ; q++) {
                    s[q] = 0.0;
#pragma unroll
                    for (int t = 0; t < kSteps; t++) s[q] += (double)cv[q * kSteps + t];
                }
                const double t = wave_sum4(s);
                if ((uint32_t)ln / kQ == j / kQ) mine = t;
#pragma unroll
                for (int q = 0; q < kQ * kSteps; q++) u[q] = nu[q];
            }
            if ((uint32_t)ln < cnt) {
                if (one) finish(hv, mine, xo, dout);
                else a.hubpart[c] = mine;
            }
        }
        // in-hubs of several chunks wait for every block's sums: arrive now,
        // wait once the other vertices are done
        grid_signal(a.bar, xcc, gen, a.abort);
        // (A2) every other vertex, a 64-vertex word per wave at a time: from
        // the sliced in-edges (each lane sums its own vertex's row entries in
        // order) or, without them, by a scheduled walk of the word's lists
        if (g.sell_src) {
            constexpr uint32_t U = 4;
            for (uint32_t first = gwave; first < W; first += nwaves * kWave) {
                const uint32_t cnt = min((uint32_t)kWave, (W - first + nwaves - 1) / nwaves);
                // a lane holds one word's rows; what a word's vertices need in
                // the end is loaded one word ahead, its in-edges one step ahead
                uint32_t off = 0, nrow = 0;
                if ((uint32_t)ln < cnt) {
                    const uint32_t w = first + (uint32_t)ln * nwaves;
                    off = g.sell_off[w];
                    nrow = (g.sell_off[w + 1] - off) / kWave;
                }
                struct Own {
                    uint32_t dout, din;
                    float xo;
                };
                auto load_own = [&](uint32_t i) {
                    Own o{0u, kPad, 0.f};
                    const uint32_t v = (first + i * nwaves) * kWave + ln;
                    if (v < n) {
                        o.dout = g.row[v + 1] - g.row[v];
                        o.din = g.cstart[v + 1] - g.cstart[v];
                        o.xo = a.x[v];
                    }
                    return o;
                };
                auto load = [&](uint32_t i, uint32_t j, uint32_t *u) {
                    const uint32_t rows = lane_value(nrow, (int)i);
                    const uint32_t *S = g.sell_src + lane_value(off, (int)i) + ln;
#pragma unroll
                    for (uint32_t q = 0; q < U; q++) {
                        u[q] = kPad;
                        if (j + q < rows) u[q] = S[(size_t)(j + q) * kWave];
                    }
                };
                uint32_t i = 0, j = 0, u[U], nu[U];
                Own own = load_own(0), next = own;
                load(0, 0, u);
                double s = 0.0;
                while (i < cnt) {
                    if (j == 0 && i + 1 < cnt) next = load_own(i + 1);
                    const uint32_t rows = lane_value(nrow, (int)i);
                    const bool last = j + U >= rows;
                    const uint32_t ni = last ? i + 1 : i, nj = last ? 0u : j + U;
                    if (ni < cnt) load(ni, nj, nu);
                    if (rows) {
                        float cv[U];
                        gather(u, cv, std::integral_constant<int, (int)U>{});
#pragma unroll
                        for (uint32_t q = 0; q < U; q++) s += (double)cv[q];
                    }
                    if (last) {
                        if (own.din <= kPullHubDegree) finish((first + i * nwaves) * kWave + ln, s, own.xo, own.dout);
                        s = 0.0;
                        own = next;
                    }
#pragma unroll
                    for (uint32_t q = 0; q < U; q++) u[q] = nu[q];
                    i = ni;
                    j = nj;
                }
            }
        } else {
            for (uint32_t w = gwave; w < W; w += nwaves) {
                const uint32_t v = w * kWave + ln;
                uint32_t b = 0, e = 0;
                bool own = false;
                if (v < n) {
                    b = g.cstart[v];
                    e = g.cstart[v + 1];
                    own = e - b <= kPullHubDegree;
                    if (!own) b = e;
                }
                const CSum s = wave_gather_csum(b, e, [&](uint32_t ed) {
                    const uint32_t u = g.csrc[ed];
                    return u < ncc ? s_cc[u] : cc[u];
                });
                if (own) finish(v, (double)s.hi + (double)s.lo, a.x[v], g.row[v + 1] - g.row[v]);
            }
        }
        // (B) in-hubs of several chunks, eight lanes each (those of more than
        // kHubWave chunks: the whole wave), dealt out so that the largest,
        // which come first, fall to different waves; the first ones' data is
        // loaded before the wait
        constexpr uint32_t kHubLanes = 8, kHubs = kWave / kHubLanes, kHubWave = 8 * kHubLanes;
        struct Hub {
            uint32_t at, chunks, v, dout;
            float xo;
        };
        auto load_hub = [&](uint32_t h0) {
            Hub b{0u, 0u, 0u, 0u, 0.f};
            const uint32_t h = h0 + (uint32_t)ln / kHubLanes * nwaves;
            if (h < g.nhubin) {
                const uint2 d = g.hubin[h];
                b.at = d.x;
                b.chunks = d.y;
                if (d.y > 1) {
                    b.v = g.hugein[d.x].x;
                    b.dout = g.row[b.v + 1] - g.row[b.v];
                    b.xo = a.x[b.v];
                }
            }
            return b;
        };
        uint32_t h0 = gwave;
        Hub hb = load_hub(h0);
        ok = grid_wait(a.bar, gen, a.abort);
        if (!ok) break;
        while (h0 < g.nhubin) {
            const Hub cur = hb;
            h0 += nwaves * kHubs;
            if (h0 < g.nhubin) hb = load_hub(h0);
            double s = 0.0;
            if (cur.chunks > 1 && cur.chunks <= kHubWave) {
#pragma unroll 8
                for (uint32_t k = (uint32_t)ln % kHubLanes; k < cur.chunks; k += kHubLanes) s += a.hubpart[cur.at + k];
            }
            s += dpp<kDppQuad1>(0.0, s);
            s += dpp<kDppQuad2>(0.0, s);
            s += dpp<kDppHalfMirror>(0.0, s);
            uint64_t wide = ballot(cur.chunks > kHubWave);
            while (wide) {
                const int l = first_lane(wide);
                const uint32_t at = lane_value(cur.at, l), chunks = lane_value(cur.chunks, l);
                double t = 0.0;
                for (uint32_t k = ln; k < chunks; k += kWave) t += a.hubpart[at + k];
                t = wave_sum_f64(t);
                if (ln / (int)kHubLanes == l / (int)kHubLanes) s = t;
                wide &= ~(0xFFull << l);
            }
            if (ln % (int)kHubLanes == 0 && cur.chunks > 1) finish(cur.v, s, cur.xo, cur.dout);
        }
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
    float *p;          // d r / outdeg of this round's active vertices [n]
    uint64_t *abit;    // 2 x W: active vertices of rounds k (k % 2)
    uint32_t *queue;   // 2 x qcap: vertices whose residual crossed theta
    uint32_t qcap;
    FrontierCtr *ctr;  // [0,1]: activation totals; [2,3,4]: queue appends
    PrPart *part;      // kMaxBlocks partials for the final sums
    GridBarrier bar;
    uint32_t *abort;
    DevStats *stats;
    DevTrace *trace;
    double damping, theta, alpha;
    double total_wl;
    int32_t force;     // -1 auto, 0 push, 1 pull
    uint32_t max_rounds;
    uint32_t probe;
    uint32_t iterative;  // rounds chosen by the ITERATIVE scheme's predicted times
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

// In-hub chunks and slice rows a wave of a residual pull round keeps in flight.
constexpr int kDdChunks = 2;
constexpr int kDdRows = 8;

struct DdRound {
    const PrDdArgs *a;
    double theta;
    Stager S;
    unsigned long long count;
    unsigned long long qscout;  // out-degree sum of queued vertices (ITERATIVE)
    bool qdeg;
};

// Add `add` to v's residual (atomically when `atomic`), queueing v if this
// addition took its residual across theta. An atomic addition returns the
// old value, so the lane recomputes the rounded sum the atomic stored and
// adds its rounding error (TwoSum, Knuth) to rlo[v]. Wave-convergent.
__device__ __forceinline__ void dd_accumulate(DdRound &R, bool act, uint32_t v, CSum add, bool atomic)
{
    bool crossed = false;
    const float ad = csum_value(add);
    if (act && ad > 0.f) {
        float old;
        if (atomic) {
            old = atomicAdd(&R.a->r[v], add.hi);
            const float s = old + add.hi;
            const float bb = s - old;
            const float err = (old - (s - bb)) + (add.hi - bb) + add.lo;
            if (err != 0.f) atomicAdd(&R.a->rlo[v], err);
        } else {
            CSum c{R.a->r[v], R.a->rlo[v]};
            old = c.hi;
            c = csum_merge(c, add);
            R.a->r[v] = c.hi;
            R.a->rlo[v] = c.lo;
        }
        crossed = (double)old < R.theta && (double)old + (double)ad >= R.theta;
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
        if (dg) pu = a.p[u];
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
        dd_accumulate(R, act, v, CSum{pk, 0.f}, true);
    }
}

template <int BS>
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

    __shared__ double s_smp[kPrioSort];
    // pull rounds test the active bits of the lowest ids (in a degree-ordered
    // graph the sources of most in-edges) in an LDS copy of the bitmap
#ifndef SG_PRDD_LDS
#define SG_PRDD_LDS 8
#endif
    constexpr uint32_t kAbLds = SG_PRDD_LDS * BS;
    __shared__ uint64_t s_ab[kAbLds];
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
    bool ok = grid_sync<true>(a.bar, xcc, gen, a.abort);
    __shared__ unsigned long long s_stamp;
    IterativePolicy ipol;
    unsigned long long stamp0 = 0, stamp_prev = 0;
    float in_wl_prev = 0.f;
    int v_prev = -1;
    bool held = false;  // the last activation held residuals >= theta back (priority)

    uint32_t k = 0, pushes = 0, pulls = 0;
    unsigned long long ptrace = 0;
    while (ok) {
        if (a.max_rounds && k >= a.max_rounds) break;
        // ---- activation: move residual >= theta into y, set p and the bit
        if (threadIdx.x == 0) s_stamp = barrier_stamp(a.bar);
        read_counts(&q_ctr[k % 3], s_lvl);
        __syncthreads();
        const RoundCounts qc = unpack_counts(s_lvl, a.qcap);
        const unsigned long long stamp = s_stamp;
        __syncthreads();
        // ITERATIVE: time the round that just ended, then pick this round's
        // variant (topology-driven ones rebuild the active set by a scan)
        int var = -1;
        if (a.iterative) {
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
            if (dout) a.p[u] = df * ru / (float)dout;
            scout += dout;
            cnt++;
        };
        bool waiting = false;  // this lane saw a residual >= theta left below the priority threshold
        // a scan also after a round that held residuals back: they did not
        // cross theta again, so no queue holds them
        // or once the queue holds an eighth of the vertices (it holds every
        // residual >= theta, so a scan finds the same set): reading all residuals
        // in order then costs less than two returning atomics per entry
        if (k == 0 || qc.overflow || held || var == kItPullTd || var == kItPushTd || qc.qlen > n / 8) {
            double thr = theta;
            if (var == kItPushTd && a.cut > 0.f) thr = fmax(theta, sampled_threshold<BS>(a, k, s_smp));
            for (uint32_t w = gwave; w < W; w += nwaves) {
                const uint32_t v = w * 64 + ln;
                bool act = false;
                if (v < n) {
                    const float rv = a.r[v] + a.rlo[v];
                    act = (double)rv >= thr;
                    waiting |= !act && (double)rv >= theta;
                    if (act) {
                        a.r[v] = 0.f;
                        a.rlo[v] = 0.f;
                        activate(v, rv);
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
                    atomicAdd(&a.r[u], hi);
                    atomicAdd(&a.rlo[u], lo);
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
        bool pull;
        if (var >= 0) pull = var == kItPullTd;
        else if (a.force >= 0) pull = a.force == 1;
        else pull = (double)ac.scout > a.total_wl / a.alpha;
        if (pull) {
            pulls++;
            if (k < 64) ptrace |= 1ull << k;
        } else {
            pushes++;
        }
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
        } else if (gtid == 0) {
            write_trace(a.trace, k, pull, ac.count, ac.scout, t_start);
        }
        if (blockIdx.x == 0) {
            clear_ctr(&act_ctr[(k + 1) & 1]);
            clear_ctr(&q_ctr[(k + 2) % 3]);
        }
        uint64_t *ab_next = a.abit + (size_t)((k + 1) & 1) * W;
        for (uint32_t w = gtid; w < W; w += nthreads) ab_next[w] = 0;

        DdRound R;
        R.a = &a;
        R.theta = theta;
        R.S = Stager{a.queue + (size_t)((k + 1) & 1) * a.qcap, a.qcap, &q_ctr[(k + 1) % 3], s_q, &s_qn, kLdsQ};
        R.count = 0;
        R.qscout = 0;
        R.qdeg = a.iterative != 0;
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
                    const float pu = a.p[u];
                    for (uint32_t e0 = beg; e0 < end; e0 += kWave) {
                        const uint32_t e = e0 + ln;
                        const bool act = e < end;
                        dd_accumulate(R, act, act ? g.col[e] : 0u, CSum{pu, 0.f}, true);
                    }
                }
            }
            for (uint32_t w = gwave; w < W; w += nwaves) {
                const uint64_t word = ab[w];
                if (word) dd_push_word(R, word, w);
            }
        } else {
            const uint32_t nab = min(W, kAbLds);
            for (uint32_t i = threadIdx.x; i < nab; i += BS) s_ab[i] = ab[i];
            __syncthreads();
            auto active = [&](uint32_t u) -> bool {
                const uint32_t w = u >> 6;
                return ((w < nab ? s_ab[w] : ab[w]) >> (u & 63)) & 1;
            };
            // in-hub chunks, kDdChunks per wave together with every load of a
            // stage issued for all of them before any is used, their sums
            // merged into the hubs by one lane each. A wave's chunks are
            // nwaves apart, so a short list still spreads over every wave.
            constexpr int kSteps = (int)(kPullChunk / kWave);
            for (uint32_t c0 = gwave; c0 < g.nhugein; c0 += nwaves * kDdChunks) {
                uint32_t cv[kDdChunks], cb[kDdChunks], ce[kDdChunks];
#pragma unroll
                for (int q = 0; q < kDdChunks; q++) {
                    const uint32_t c = c0 + (uint32_t)q * nwaves;
                    cv[q] = cb[q] = ce[q] = 0;
                    if (c < g.nhugein) {
                        const uint2 dsc = g.hugein[c];
                        cv[q] = dsc.x;
                        cb[q] = dsc.y;
                        ce[q] = min(g.cstart[dsc.x + 1], dsc.y + kPullChunk);
                    }
                }
                uint32_t u[kDdChunks][kSteps];
#pragma unroll
                for (int q = 0; q < kDdChunks; q++)
#pragma unroll
                    for (int t = 0; t < kSteps; t++) {
                        const uint32_t e = cb[q] + (uint32_t)(t * kWave + ln);
                        u[q][t] = e < ce[q] ? g.csrc[e] : 0xFFFFFFFFu;
                    }
                float pu[kDdChunks][kSteps];
#pragma unroll
                for (int q = 0; q < kDdChunks; q++)
#pragma unroll
                    for (int t = 0; t < kSteps; t++)
                        pu[q][t] = u[q][t] != 0xFFFFFFFFu && active(u[q][t]) ? a.p[u[q][t]] : 0.f;
                uint32_t hv = 0;
                CSum hs{0.f, 0.f};
#pragma unroll
                for (int q = 0; q < kDdChunks; q++) {
                    CSum s{0.f, 0.f};
#pragma unroll
                    for (int t = 0; t < kSteps; t++) csum_add(s, pu[q][t]);
                    s = wave_csum(s);
                    if (ln == q) {
                        hv = cv[q];
                        hs = s;
                    }
                }
                dd_accumulate(R, ln < kDdChunks, hv, hs, true);
            }
            for (uint32_t w = gwave; w < W; w += nwaves) {
                const uint32_t v = w * 64 + ln;
                uint32_t b = 0, e = 0;
                bool own = false;
                if (v < n) {
                    b = g.cstart[v];
                    e = g.cstart[v + 1];
                    own = e - b <= kPullHubDegree;
                    if (!own) b = e;
                }
                CSum s{0.f, 0.f};
                if (g.sell_src) {
                    // by the sliced in-edges, a lane per vertex: its sum stays
                    // in registers, with no edge scheduling and no segmented
                    // scans. RMAT graph of 100 003 vertices, 1.4 M edges,
                    // nearly all active: 95 -> 45 us a round, 9.6 -> 4.8 ms a run
                    // (rows in flight 4, 8, 16: within 5 %)
                    const uint32_t beg = g.sell_off[w];
                    const uint32_t rows = (g.sell_off[w + 1] - beg) / kWave;
                    const uint32_t *S = g.sell_src + beg + ln;
                    const uint32_t deg = e - b;
                    for (uint32_t j0 = 0; j0 < rows; j0 += kDdRows) {
                        uint32_t u[kDdRows];
                        float pu[kDdRows];
#pragma unroll
                        for (int q = 0; q < kDdRows; q++)
                            u[q] = j0 + q < deg ? S[(size_t)(j0 + q) * kWave] : 0xFFFFFFFFu;
#pragma unroll
                        for (int q = 0; q < kDdRows; q++)
                            pu[q] = u[q] != 0xFFFFFFFFu && active(u[q]) ? a.p[u[q]] : 0.f;
#pragma unroll
                        for (int q = 0; q < kDdRows; q++) csum_add(s, pu[q]);
                    }
                } else {
                    s = wave_gather_csum(b, e, [&](uint32_t ed) {
                        const uint32_t u = g.csrc[ed];
                        return active(u) ? a.p[u] : 0.f;
                    });
                }
                dd_accumulate(R, own, v, s, false);
            }
        }
        publish_counts<WPB>(&q_ctr[(k + 1) % 3], R.qscout, R.count, false, s_red);
        flush_stage(R.S, s_flush);
        k++;
        ok = grid_sync<true>(a.bar, xcc, gen, a.abort);
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
        if (threadIdx.x == 0) a.part[blockIdx.x] = t;
        ok = grid_sync(a.bar, xcc, gen, a.abort);
    }
    PrPart tot{0.0, 1.f, 0.f};
    if (ok) {
        tot = grid_part<BS>(a.part, gridDim.x, s_red2, &s_glob);
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
        a.hubpart = (double *)(base + off_hub);
        a.part = (double2 *)(base + off_part);
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
        // y (n compensated floats) | r | rlo | p (n floats each) | partials
        const uint64_t off_part = (n * 8 + 3 * n * 4 + 15) / 16 * 16;
        if ((rc = engine_ensure_aux(e, off_part + part_bytes))) return rc;
        char *base = (char *)e->aux;
        PrDdArgs a{};
        a.g = d;
        a.x = (float *)res;
        a.y = (CSum *)base;
        a.r = (float *)(base + n * 8);
        a.rlo = (float *)(base + n * 12);
        a.p = (float *)(base + n * 16);
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
        a.iterative = mode == SG_PR_ITERATIVE;
        a.it_force = it_force;
        a.ticks_per_us = (float)(e->wall_khz / 1000.0);
        a.cut = 0.f;
        if (mode == SG_PR_ITERATIVE && o.priority == SG_PRIO_SAMPLING) {
            if (!(o.cut_threshold > 0.f && o.cut_threshold < 1.f))
                SG_FAIL(SG_ERR_RANGE, "sg_pagerank: sample-based priority needs 0 < cut_threshold < 1");
            a.cut = o.cut_threshold;
        }
        switch (bs) {
        case 256: rc = launch_persistent<PrDdArgs, k_pr_dd<256>>(e, a, 256); break;
        case 512: rc = launch_persistent<PrDdArgs, k_pr_dd<512>>(e, a, 512); break;
        default: rc = launch_persistent<PrDdArgs, k_pr_dd<1024>>(e, a, 1024); break;
        }
    }
    if (rc) return rc;
    if ((rc = engine_finish(e, 1))) return rc;
    e->timed = true;
    e->clocked = e->last_grid;
    return SG_OK;
}
