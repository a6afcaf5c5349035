// Betweenness centrality (Brandes) for up to 64 sources per launch, one
// persistent kernel per batch.
//
// Reference path: samples/hybrid_bc/hybrid_bc.cu. Stage 1 (the BC app,
// hybrid_bc.cu:23-131) runs the hybrid BFS engine accumulating path counts
// sigma and pushes each level's vertices onto a WorklistStack
// (include/framework/worklist_stack.cuh:16-111); stage 2 (StageTwoDDFused,
// hybrid_bc.cu:134-225) walks the stack back level by level adding
// sigma(v)/sigma(w) (1 + delta(w)) over successors w; the result is halved
// (hybrid_bc.cu:374-376). The reference handles one source per run, with
// sigma and delta in FP32.
//
// Here a batch of B <= 64 sources shares every traversal of the adjacency:
//   * each vertex carries 64-bit masks, bit s for source s: `seen` and one
//     mask per BFS level (a ring of three dense n-word arrays);
//   * per-source state is laid out source-minor, [vertex][64], so a wave
//     handles one vertex with lane s = source s and reads a neighbour's row
//     (512 B of sigma or psi) as one coalesced access;
//   * the forward pass is level-synchronous: discovery of the next level's
//     masks (push over the level's out-edges with atomicOr, or pull over
//     in-edges of vertices not yet seen by every source, switched by the
//     alpha rule on the level's out-degree), then sigma of every newly
//     reached (vertex, source) pair gathered from its predecessors on that
//     level (FP64, no atomics except for in-hubs split into chunks);
//   * every (vertex, level-mask) pair is pushed on a level stack, so the
//     backward pass visits each vertex once per distinct depth it has over
//     the batch;
//   * the backward pass stores psi(w) = (1 + delta(w)) / sigma(w) per
//     (vertex, source), so a predecessor v needs one load per successor:
//     delta(v) = sigma(v) * sum of psi(w) over successors w. delta is FP64 in
//     registers; bc(v) += delta(v) / 2 accumulates in FP64 over batches and
//     is written out as FP32.
#include "frontier.hpp"

using namespace sg;

namespace {

constexpr uint32_t kMaxLevels = 1u << 20;

// First element of source s's result row: rows are n elements, and `orow`
// (when given) maps a batch's sources onto rows of a larger result pool.
__device__ __forceinline__ size_t out_row(const uint32_t *orow, uint32_t s, uint32_t n)
{
    return (size_t)(orow ? orow[s] : s) * n;
}

// A batch's sources: handed to the kernel as arguments, or already on the device.
struct MsSources {
    const uint32_t *dev;
    uint32_t v[64];
    __device__ __forceinline__ uint32_t get(int i) const { return dev ? dev[i] : v[i]; }
};

struct BcArgs {
    DevGraph g;
    MsSources src;        // sources of this batch
    uint32_t nsrc;
    uint64_t *seen;       // [n]
    uint64_t *F;          // 3 x n: level masks, level L in F + (L % 3) n
    double *sigma;        // [n][64]
    double *psi;          // [n][64]
    double *bc;           // [n], FP64 accumulator over batches
    float *out;           // [n], written by the last batch
    float *dep;           // optional: 0.5 delta_s(v) in row out_row(orow, s) of n floats
    const uint32_t *orow; // optional result row of each source (null: row s)
    uint32_t *stk_v;      // level stack: vertex
    uint64_t *stk_m;      // level stack: sources with that vertex at this level
    uint32_t cap;
    uint32_t *lvl;        // stack start of each level [kMaxLevels + 2]
    uint32_t *ctl;        // [0] stack length, [1] overflow
    FrontierCtr *ctr;     // 3 slots: per-level entry count / out-degree sum
    GridBarrier bar;
    uint32_t *abort;
    DevStats *stats;
    DevTrace *trace;
    double alpha, beta;
    double total_wl;
    int32_t force;
    uint32_t first, last;
    uint32_t probe;
};

__device__ __forceinline__ uint64_t wave_or_u64(uint64_t x)
{
    return wave_reduce(x, (uint64_t)0, [](uint64_t a, uint64_t b) { return a | b; });
}

__device__ __forceinline__ uint64_t seg_or(uint64_t s, int k)
{
    return wave_seg_scan(s, (uint32_t)k, [](uint64_t a, uint64_t b) { return a | b; });
}

// OR over in-edges [b, e) of each lane's vertex of Fc[csrc[edge]], the wave
// walking the concatenated lists 64 edges per step. A lane stops once its OR
// holds every bit of `need` (the reference's early break, generalised to a
// set of sources: with one source it stops at the first parent).
__device__ __forceinline__ uint64_t wave_gather_or(const DevGraph &g, const uint64_t *Fc, uint32_t b, uint32_t e,
                                                   uint64_t need)
{
    const int ln = lane();
    uint64_t acc = 0;
    for (;;) {
        const uint32_t r = e - b;
        const uint32_t incl = wave_incl_scan(r);
        const uint32_t total = lane_value(incl, kWave - 1);
        if (total == 0) break;
        const uint32_t excl = incl - r;
        const uint32_t j = (uint32_t)ln;
        const int k = owner_lane(incl, j);
        const uint32_t bk = shfl(b, k), xk = shfl(excl, k);
        uint64_t cand = 0;
        if (j < total) cand = Fc[g.csrc[bk + (j - xk)]];
        const uint64_t s = seg_or(cand, k);
        const uint32_t lo = min(excl, 64u), hi = min(incl, 64u), cov = hi - lo;
        const uint64_t seg = __shfl(s, (int)(hi > 0 ? hi - 1 : 0), kWave);
        if (cov) {
            acc |= seg;
            b += cov;
            if ((acc & need) == need) b = e;
        }
    }
    return acc;
}

// Rows a wave loads before it adds any: a row's load is a trip to L2 or
// memory, and one at a time they made a vertex's sum a serial chain. 64-source
// BC on an RMAT graph of 65 536 vertices: 2224 us one at a time, 1653 with eight.
constexpr int kRowsInFlight = 8;

// Sum, in lane s, of row[u][s] over the edges [b, e) (edge ids into `adj`)
// whose neighbour u has bit s in (M[u] & mask). Whole wave, uniform b/e/mask.
__device__ __forceinline__ double masked_row_sum(const uint32_t *adj, const uint64_t *M, const double *row,
                                                 uint32_t b, uint32_t e, uint64_t mask)
{
    const int ln = lane();
    double acc = 0.0;
    for (uint32_t e0 = b; e0 < e; e0 += kWave) {
        const uint32_t ed = e0 + ln;
        uint32_t u = 0;
        uint64_t fm = 0;
        if (ed < e) {
            u = adj[ed];
            fm = M[u] & mask;
        }
        uint64_t mm = ballot(fm != 0);
        uint64_t srcs = wave_or_u64(fm);
        if (__popcll(srcs) < __popcll(mm)) {
            // fewer sources than matching neighbours (small batches): per
            // source, every lane loads its neighbour's value and the wave sums
            while (srcs) {
                int s[kRowsInFlight];
                double x[kRowsInFlight];
#pragma unroll
                for (int q = 0; q < kRowsInFlight; q++) {
                    s[q] = srcs ? first_lane(srcs) : -1;
                    srcs &= srcs - 1;
                    x[q] = s[q] >= 0 && ((fm >> s[q]) & 1) ? row[(size_t)u * 64 + s[q]] : 0.0;
                }
#pragma unroll
                for (int q = 0; q < kRowsInFlight; q++) {
                    if (s[q] < 0) break;  // wave-uniform
                    const double sum = wave_sum_f64(x[q]);
                    if (ln == s[q]) acc += sum;
                }
            }
            continue;
        }
        while (mm) {
            double x[kRowsInFlight];
#pragma unroll
            for (int q = 0; q < kRowsInFlight; q++) {
                x[q] = 0.0;
                if (!mm) continue;  // wave-uniform
                const int j = first_lane(mm);
                mm &= mm - 1;
                const uint64_t fj = lane_value(fm, j);
                const uint32_t uj = lane_value(u, j);
                if ((fj >> ln) & 1) x[q] = row[(size_t)uj * 64 + ln];
            }
#pragma unroll
            for (int q = 0; q < kRowsInFlight; q++) acc += x[q];
        }
    }
    return acc;
}

// Slice rows a wave of a pull discovery keeps in flight.
constexpr int kDiscoverRows = 8;

// Discovery of the next level's masks: Fn[w] gets the bits of sources that
// reach w for the first time through a level-L vertex. Push expands the
// level's entries (seg_v/seg_m, len) over out-edges with atomicOr; pull has
// every vertex not yet seen by all sources OR its in-neighbours' level masks.
// Whole grid; `seen` holds every level up to L.
__device__ __forceinline__ void ms_discover(const DevGraph &g, const uint64_t *seen, const uint64_t *Fc, uint64_t *Fn,
                                            const uint32_t *seg_v, const uint64_t *seg_m, uint32_t len, uint64_t bm,
                                            bool pull, uint32_t gwave, uint32_t nwaves)
{
    const int ln = lane();
    const uint32_t n = g.n, W = g.words;
    if (!pull) {
        for (uint32_t c0 = 0; c0 < g.nhuge; c0 += nwaves * kWave) {
            const uint32_t c = c0 + (uint32_t)ln * nwaves + gwave;
            uint2 dsc = make_uint2(0u, 0u);
            uint64_t mk = 0;
            if (c < g.nhuge) {
                dsc = g.huge[c];
                mk = Fc[dsc.x];
            }
            uint64_t mm = ballot(mk != 0);
            while (mm) {
                const int t = first_lane(mm);
                mm &= mm - 1;
                const uint32_t u = lane_value(dsc.x, t), beg = lane_value(dsc.y, t);
                const uint64_t mu = lane_value(mk, t);
                const uint32_t end = min(g.row[u + 1], beg + kHugeChunk);
                for (uint32_t e0 = beg; e0 < end; e0 += kWave) {
                    const uint32_t e = e0 + ln;
                    if (e < end) {
                        const uint32_t w = g.col[e];
                        const uint64_t nm = mu & ~seen[w];
                        if (nm && (Fn[w] & nm) != nm) atomicOr((unsigned long long *)&Fn[w], (unsigned long long)nm);
                    }
                }
            }
        }
        const uint32_t per = (len + nwaves - 1) / nwaves;
        const uint32_t qb = min(len, gwave * per), qe = min(len, gwave * per + per);
        for (uint32_t i0 = qb; i0 < qe; i0 += kWave) {
            const uint32_t i = i0 + ln;
            uint32_t b = 0, d = 0;
            uint64_t mu = 0;
            if (i < qe) {
                const uint32_t u = seg_v[i];
                mu = seg_m[i];
                b = g.row[u];
                d = g.row[u + 1] - b;
                if (d > kHugeDegree) d = 0;
            }
            const uint32_t incl = wave_incl_scan(d);
            const uint32_t total = lane_value(incl, kWave - 1);
            const uint32_t off = b - (incl - d);
            for (uint32_t jb = 0; jb < total; jb += kWave) {
                const uint32_t j = jb + ln;
                const int k = owner_lane(incl, j);
                const uint32_t e = shfl(off, k) + j;
                const uint64_t mk = __shfl(mu, k, kWave);
                if (j < total) {
                    const uint32_t w = g.col[e];
                    const uint64_t nm = mk & ~seen[w];
                    if (nm && (Fn[w] & nm) != nm) atomicOr((unsigned long long *)&Fn[w], (unsigned long long)nm);
                }
            }
        }
    } else {
        for (uint32_t c = gwave; c < g.nhugein; c += nwaves) {
            const uint2 dsc = g.hugein[c];
            const uint64_t unseen = bm & ~seen[dsc.x];
            if (!unseen) continue;
            const uint32_t end = min(g.cstart[dsc.x + 1], dsc.y + kPullChunk);
            constexpr int K = (int)(kPullChunk / kWave);
            uint32_t u[K];
            uint64_t f[K], o = 0;
#pragma unroll
            for (int k = 0; k < K; k++) {
                const uint32_t e = dsc.y + (uint32_t)(k * kWave + ln);
                u[k] = e < end ? g.csrc[e] : 0xFFFFFFFFu;
            }
#pragma unroll
            for (int k = 0; k < K; k++) f[k] = u[k] != 0xFFFFFFFFu ? Fc[u[k]] : 0ull;
#pragma unroll
            for (int k = 0; k < K; k++) o |= f[k];
            o = wave_or_u64(o) & unseen;
            if (ln == 0 && o) atomicOr((unsigned long long *)&Fn[dsc.x], (unsigned long long)o);
        }
        // By the sliced in-edges, a lane per vertex and kDiscoverRows rows in
        // flight, a lane stopping once it has every bit it lacks: a vertex's
        // OR stays in a register, where scheduling the edges over the wave
        // took a segmented 64-bit scan per 64 of them. A graph with fewer
        // words than waves gives each word to `parts` waves, which take its rows
        // in turn and merge by atomics. 64 BFS on an RMAT graph of 524 288
        // vertices: its pull rounds 212, 204, 161, 77, 32 us by scheduled edges
        // and an append atomic per word, 108, 101, 59, 31, 26 by rows and
        // append_level.
        if (g.sell_src) {
            uint32_t parts = 1;
            while (parts < 16 && (uint64_t)parts * 2 * W <= nwaves) parts <<= 1;
            for (uint32_t it = gwave; it < W * parts; it += nwaves) {
                const uint32_t w = it / parts, part = it % parts, v = w * 64 + (uint32_t)ln;
                uint64_t unseen = 0, acc = 0;
                uint32_t deg = 0;
                if (v < n) {
                    unseen = bm & ~seen[v];
                    deg = g.cstart[v + 1] - g.cstart[v];
                    if (deg > kPullHubDegree) deg = 0;
                }
                uint32_t j0 = part * kDiscoverRows;
                bool act = unseen && j0 < deg;
                if (!ballot(act)) continue;
                const uint32_t *S = g.sell_src + g.sell_off[w] + ln;
                for (; ballot(act); j0 += parts * kDiscoverRows) {
                    uint32_t u[kDiscoverRows];
                    uint64_t f[kDiscoverRows];
#pragma unroll
                    for (int k = 0; k < kDiscoverRows; k++)
                        u[k] = act && j0 + k < deg ? S[(size_t)(j0 + k) * kWave] : 0xFFFFFFFFu;
#pragma unroll
                    for (int k = 0; k < kDiscoverRows; k++) f[k] = u[k] != 0xFFFFFFFFu ? Fc[u[k]] : 0ull;
#pragma unroll
                    for (int k = 0; k < kDiscoverRows; k++) acc |= f[k];
                    act = act && j0 + parts * kDiscoverRows < deg && (acc & unseen) != unseen;
                }
                acc &= unseen;
                if (acc && parts == 1) Fn[v] = acc;
                else if (acc) atomicOr((unsigned long long *)&Fn[v], (unsigned long long)acc);
            }
            return;
        }
        for (uint32_t w = gwave; w < W; w += nwaves) {
            const uint32_t v = w * 64 + ln;
            uint32_t b = 0, e = 0;
            uint64_t unseen = 0;
            if (v < n) {
                unseen = bm & ~seen[v];
                b = g.cstart[v];
                e = g.cstart[v + 1];
                if (!unseen || e - b > kPullHubDegree) b = e;
            }
            const uint64_t o = wave_gather_or(g, Fc, b, e, unseen) & unseen;
            if (o) Fn[v] = o;
        }
    }
}

// Appends (v, F[v]) of every vertex with a bit in F to the pair list (vv, mm)
// whose length is *count, one atomic per block (one per word of vertices, all
// on the same counter, serialise at 11 ns each: 90 us a level on 2^19
// vertices): the block's waves count first, then write. s_at: WPB words. Past
// `cap` entries *overflow is set.
template <int WPB>
__device__ __forceinline__ void append_level(const uint64_t *F, uint32_t n, uint32_t W, uint32_t gwave, uint32_t nwaves,
                                             uint32_t *count, uint32_t *vv, uint64_t *mm, uint32_t cap,
                                             uint32_t *overflow, uint32_t *s_at)
{
    const int ln = lane(), wid = threadIdx.x / kWave;
    uint32_t mine = 0;
    for (uint32_t w = gwave; w < W; w += nwaves) {
        const uint32_t v = w * 64 + (uint32_t)ln;
        mine += (uint32_t)__popcll(ballot(v < n && F[v] != 0));
    }
    if (ln == 0) s_at[wid] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t sum = 0;
        for (int i = 0; i < WPB; i++) sum += s_at[i];
        uint32_t at = sum ? atomicAdd(count, sum) : 0u;
        for (int i = 0; i < WPB; i++) {
            const uint32_t c = s_at[i];
            s_at[i] = at;
            at += c;
        }
    }
    __syncthreads();
    uint32_t at = s_at[wid];
    if (!mine) return;
    for (uint32_t w = gwave; w < W; w += nwaves) {
        const uint32_t v = w * 64 + (uint32_t)ln;
        const uint64_t x = v < n ? F[v] : 0ull;
        const uint64_t m = ballot(x != 0);
        if (x) {
            const uint32_t pos = at + (uint32_t)rank_in(m);
            if (pos < cap) {
                vv[pos] = v;
                mm[pos] = x;
            } else {
                *overflow = 1;
            }
        }
        at += (uint32_t)__popcll(m);
    }
}

// Append (v, m) for lanes with `pred` to the pair list (vv, mm) whose length
// is *count (one atomic per wave); past `cap` entries *overflow is set.
__device__ __forceinline__ void append_pair(uint32_t *count, uint32_t *vv, uint64_t *mm, uint32_t cap,
                                            uint32_t *overflow, bool pred, uint32_t v, uint64_t m)
{
    const uint64_t bm = ballot(pred);
    if (!bm) return;
    const int leader = first_lane(bm);
    uint32_t base = 0;
    if (lane() == leader) base = atomicAdd(count, (uint32_t)__popcll(bm));
    base = lane_value(base, leader);
    if (pred) {
        const uint32_t pos = base + rank_in(bm);
        if (pos < cap) {
            vv[pos] = v;
            mm[pos] = m;
        } else {
            *overflow = 1;
        }
    }
}

template <int BS>
__global__ __launch_bounds__(BS) void k_bc(BcArgs a)
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
    const uint64_t bm = a.nsrc >= 64 ? ~0ull : ((1ull << a.nsrc) - 1);

    __shared__ unsigned long long s_red[2][WPB];
    __shared__ unsigned long long s_lvl[5];
    __shared__ uint32_t s_len, s_at[WPB];

    // ---- prologue: clear masks; zero the rows hub chunks accumulate into
    for (uint32_t v = gtid; v < n; v += nthreads) {
        a.seen[v] = 0;
        a.F[v] = 0;
        a.F[(size_t)n + v] = 0;
        a.F[2 * (size_t)n + v] = 0;
        if (a.first) a.bc[v] = 0.0;
    }
    if (a.dep)
        for (uint32_t s = 0; s < a.nsrc; s++) {
            float *row = a.dep + out_row(a.orow, s, n);
            for (uint32_t v = gtid; v < n; v += nthreads) row[v] = 0.0f;
        }
    for (uint32_t h = gwave; h < g.nhubin; h += nwaves) a.sigma[(size_t)g.hugein[g.hubin[h].x].x * 64 + ln] = 0.0;
    for (uint32_t c = gwave; c < g.nhuge; c += nwaves) a.psi[(size_t)g.huge[c].x * 64 + ln] = 0.0;
    if (blockIdx.x == 0) {
        clear_ctr(&a.ctr[0]);
        clear_ctr(&a.ctr[1]);
        clear_ctr(&a.ctr[2]);
        if (threadIdx.x == 0) {
            a.ctl[0] = 0;
            a.ctl[1] = 0;
        }
    }
    bool ok = grid_sync(a.bar, xcc, gen, a.abort);
    if (ok && blockIdx.x == 0 && threadIdx.x < kWave) {
        // sources: lane s owns source s; a vertex listed twice gets both bits
        const bool has = (uint32_t)ln < a.nsrc;
        const uint32_t v = has ? a.src.get(ln) : 0u;
        uint64_t m = 0;
        int firstl = 64;
        for (int t = 0; t < 64; t++) {
            const uint32_t vt = lane_value(v, t);
            if (has && (uint32_t)t < a.nsrc && vt == v) {
                m |= 1ull << t;
                firstl = min(firstl, t);
            }
        }
        const bool lead = has && firstl == ln;
        if (has) a.sigma[(size_t)v * 64 + ln] = 1.0;
        if (lead) {
            a.seen[v] = m;
            a.F[v] = m;
        }
        append_pair(&a.ctl[0], a.stk_v, a.stk_m, a.cap, &a.ctl[1], lead, v, m);
        const uint32_t dv = lead ? g.row[v + 1] - g.row[v] : 0u;
        const unsigned long long sc = wave_sum_u64(dv);
        const unsigned long long cn = wave_sum_u64(lead ? 1ull : 0ull);
        if (ln == 0) {
            a.ctr[0].stripe[0].scout = sc;
            a.ctr[0].stripe[0].count = cn;
            a.lvl[0] = 0;
        }
    }
    if (ok) ok = grid_sync(a.bar, xcc, gen, a.abort);

    // ---- forward: levels 0, 1, ...
    uint32_t L = 0, prev_beg = 0, seg_beg = 0, seg_end = 0;
    uint32_t pushes = 0, pulls = 0;
    unsigned long long ptrace = 0;
    DirectionPolicy pol{a.alpha, a.beta, (uint32_t)min(a.total_wl, 4294967295.0), n, a.force};
    while (ok) {
        read_counts(&a.ctr[L % 3], s_lvl);
        if (threadIdx.x == 0) s_len = __hip_atomic_load(&a.ctl[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        const RoundCounts rc = unpack_counts(s_lvl, 0xFFFFFFFFu);
        seg_end = min(s_len, a.cap);
        __syncthreads();
        if (rc.count == 0 || L + 1 >= kMaxLevels) break;
        if (gtid == 0) a.lvl[L + 1] = seg_end;
        const bool pull = pol.next(L, rc.count, rc.scout);
        if (pull) {
            pulls++;
            if (L < 64) ptrace |= 1ull << L;
        } else {
            pushes++;
        }
        if (gtid == 0) write_trace(a.trace, L, pull, rc.count, rc.scout, t_start);
        if (blockIdx.x == 0) clear_ctr(&a.ctr[(L + 2) % 3]);
        const uint64_t *Fc = a.F + (size_t)(L % 3) * n;
        uint64_t *Fn = a.F + (size_t)((L + 1) % 3) * n;
        uint64_t *Ff = a.F + (size_t)((L + 2) % 3) * n;
        // level L-1's masks are no longer read: clear them for level L+2
        for (uint32_t i = prev_beg + gtid; i < seg_beg; i += nthreads) Ff[a.stk_v[i]] = 0;

        // (1) discovery of level L+1
        ms_discover(g, a.seen, Fc, Fn, a.stk_v + seg_beg, a.stk_m + seg_beg, seg_end - seg_beg, bm, pull, gwave, nwaves);
        ok = grid_sync(a.bar, xcc, gen, a.abort);
        if (!ok) break;

        // (2) the new level: seen, stack, sigma from predecessors on level L
        unsigned long long scout = 0, cnt = 0;
        append_level<WPB>(Fn, n, W, gwave, nwaves, &a.ctl[0], a.stk_v, a.stk_m, a.cap, &a.ctl[1], s_at);
        for (uint32_t w = gwave; w < W; w += nwaves) {
            const uint32_t v = w * 64 + ln;
            const uint64_t nw = v < n ? Fn[v] : 0ull;
            if (nw) {
                a.seen[v] |= nw;
                scout += g.row[v + 1] - g.row[v];
                cnt++;
            }
        }
        // a wave sums one vertex at a time: a graph with fewer words than
        // waves gives each word's vertices to `parts` waves (2^16 vertices, 64
        // sources: 1024 words had kept three of four waves idle)
        uint32_t parts = 1;
        while (parts < 64 && (uint64_t)parts * 2 * W <= nwaves) parts <<= 1;
        const uint32_t span = 64 / parts;
        for (uint32_t it = gwave; it < W * parts; it += nwaves) {
            const uint32_t w = it / parts, first = it % parts * span;
            const uint32_t v = w * 64 + ln;
            const bool in = (uint32_t)ln - first < span && v < n;
            uint64_t nw = 0;
            uint32_t b = 0, e = 0;
            if (in) nw = Fn[v];
            if (nw) {
                b = g.cstart[v];
                e = g.cstart[v + 1];
            }
            uint64_t cand = ballot(nw != 0 && e - b <= kPullHubDegree);
            while (cand) {
                const int t = first_lane(cand);
                cand &= cand - 1;
                const uint32_t vt = w * 64 + t;
                const uint64_t mt = lane_value(nw, t);
                const double s = masked_row_sum(g.csrc, Fc, a.sigma, lane_value(b, t), lane_value(e, t), mt);
                if ((mt >> ln) & 1) a.sigma[(size_t)vt * 64 + ln] = s;
            }
        }
        for (uint32_t c = gwave; c < g.nhugein; c += nwaves) {
            const uint2 dsc = g.hugein[c];
            const uint64_t nw = Fn[dsc.x];
            if (!nw) continue;
            const uint32_t end = min(g.cstart[dsc.x + 1], dsc.y + kPullChunk);
            const double s = masked_row_sum(g.csrc, Fc, a.sigma, dsc.y, end, nw);
            if (s != 0.0) atomicAdd(&a.sigma[(size_t)dsc.x * 64 + ln], s);
        }
        publish_counts<WPB>(&a.ctr[(L + 1) % 3], scout, cnt, false, s_red);
        pol.pull_prev = pull;
        prev_beg = seg_beg;
        seg_beg = seg_end;
        L++;
        ok = grid_sync(a.bar, xcc, gen, a.abort);
    }
    // levels 0 .. D hold entries; lvl[D + 1] is the stack length
    const uint32_t D = L ? L - 1 : 0;
    const uint32_t levels = L;

    // ---- backward: levels D .. 1
    for (uint32_t l = D; ok && l >= 1; l--) {
        const uint32_t sb = a.lvl[l], se = a.lvl[l + 1];
        const uint64_t *An = a.F + (size_t)((l + 1) % 3) * n;  // level l+1
        const uint64_t *Ac = a.F + (size_t)(l % 3) * n;        // level l
        uint64_t *Af = a.F + (size_t)((l + 2) % 3) * n;        // level l+2, then l-1
        if (l + 2 <= D) {
            const uint32_t fb = a.lvl[l + 2], fe = a.lvl[l + 3];
            for (uint32_t i = fb + gtid; i < fe; i += nthreads) Af[a.stk_v[i]] = 0;
        }
        // (the entry after next and the next one's edge range are read while
        // this one is summed)
        uint32_t i = sb + gwave;
        uint32_t v1 = i < se ? a.stk_v[i] : 0u, v2 = i + nwaves < se ? a.stk_v[i + nwaves] : 0u;
        uint32_t rb1 = g.row[v1], re1 = g.row[v1 + 1];
        uint64_t mv1 = i < se ? a.stk_m[i] : 0ull;
        for (; i < se; i += nwaves) {
            const uint32_t v = v1, rb = rb1, re = re1;
            const uint64_t mv = mv1;
            v1 = v2;
            v2 = i + 2 * nwaves < se ? a.stk_v[i + 2 * nwaves] : 0u;
            rb1 = g.row[v1];
            re1 = g.row[v1 + 1];
            mv1 = i + nwaves < se ? a.stk_m[i + nwaves] : 0ull;
            if (re - rb > kHugeDegree) continue;
            const double acc = masked_row_sum(g.col, An, a.psi, rb, re, mv);
            double dl = 0.0;
            if ((mv >> ln) & 1) {
                const double sg = a.sigma[(size_t)v * 64 + ln];
                dl = sg * acc;
                a.psi[(size_t)v * 64 + ln] = (1.0 + dl) / sg;
                if (a.dep) a.dep[out_row(a.orow, ln, n) + v] = (float)(0.5 * dl);
            }
            dl = wave_sum_f64(dl);
            if (ln == 0) a.bc[v] += 0.5 * dl;
        }
        for (uint32_t c = gwave; c < g.nhuge; c += nwaves) {
            const uint2 dsc = g.huge[c];
            const uint64_t mv = Ac[dsc.x];
            if (!mv) continue;
            const uint32_t end = min(g.row[dsc.x + 1], dsc.y + kHugeChunk);
            const double acc = masked_row_sum(g.col, An, a.psi, dsc.y, end, mv);
            if (acc != 0.0) atomicAdd(&a.psi[(size_t)dsc.x * 64 + ln], acc);
        }
        ok = grid_sync(a.bar, xcc, gen, a.abort);
        if (!ok) break;
        for (uint32_t i = sb + gwave; i < se; i += nwaves) {
            const uint32_t v = a.stk_v[i];
            if (g.row[v + 1] - g.row[v] <= kHugeDegree) continue;
            const uint64_t mv = a.stk_m[i];
            double dl = 0.0;
            if ((mv >> ln) & 1) {
                const size_t k = (size_t)v * 64 + ln;
                const double sg = a.sigma[k];
                dl = sg * a.psi[k];
                a.psi[k] = (1.0 + dl) / sg;
                if (a.dep) a.dep[out_row(a.orow, ln, n) + v] = (float)(0.5 * dl);
            }
            dl = wave_sum_f64(dl);
            if (ln == 0) a.bc[v] += 0.5 * dl;
        }
        {
            const uint32_t pb = a.lvl[l - 1], pe = a.lvl[l];
            for (uint32_t i = pb + gtid; i < pe; i += nthreads) Af[a.stk_v[i]] = a.stk_m[i];
        }
        ok = grid_sync(a.bar, xcc, gen, a.abort);
    }
    if (ok && a.last) {
        for (uint32_t v = gtid; v < n; v += nthreads) a.out[v] = (float)a.bc[v];
    }
    if (gtid == 0) {
        DevStats s = a.first ? DevStats{} : *a.stats;
        s.rounds += levels;
        s.push_rounds += pushes;
        s.pull_rounds += pulls;
        s.trace = ptrace;
        s.max_depth = max(s.max_depth, D);
        s.iterations += 1;
        const bool overflow = a.ctl[1] != 0;
        if (s.status == SG_OK) s.status = !ok ? SG_ERR_TIMEOUT : (overflow || levels + 1 >= kMaxLevels) ? SG_ERR_CAPACITY : SG_OK;
        *a.stats = s;
    }
    bar_end(a.bar);
}

// ------------------------------------------------------------ multi-source BFS
// Levels of up to 64 independent BFS queries in one launch: the discovery of
// the BC forward pass (shared masks, one adjacency sweep per level for every
// query) with each newly reached (vertex, source) pair writing its level into
// that source's own int32 row, so each query's result is a contiguous n-vector
// equal to a single-source BFS from it. Level entries live in a two-half ring
// (each vertex appears at most once per level).
struct MsBfsArgs {
    DevGraph g;
    MsSources src;
    uint32_t first;       // start the summary (else: add to it)
    uint32_t nsrc;
    uint64_t *seen;       // [n]
    uint64_t *F;          // 3 x n level masks
    int32_t *out;         // levels of source s in row out_row(orow, s), -1 when unreached
    const uint32_t *orow;
    uint8_t *lev;         // optional (with inv): level rows [n][lev_row(nsrc)], see LevelRows
    const uint32_t *inv;  // optional: out is in the caller's order, vertex v there is inv[v] here
    const uint32_t *perm; // (with inv) its inverse
    uint32_t *ring_v;     // 2 x n: entries of level L in half L % 2
    uint64_t *ring_m;
    uint32_t *ctl;        // [1] overflow, [2 + h] entries in ring half h
    FrontierCtr *ctr;
    GridBarrier bar;
    uint32_t *abort;
    DevStats *stats;
    DevTrace *trace;
    double alpha, beta;
    double total_wl;
    int32_t force;
    uint32_t max_rounds;
    uint32_t probe;
};

// Levels in the caller's order, when that is another than the device's. A pass
// over the finished rows that gathers them by `inv` reads 4 bytes from a line
// of its own per level: RMAT-19, 64 sources, 100 of 533 us. Instead the levels
// are kept as a row of bytes per vertex, one per source, and the kernel ends by
// reading whole rows in the caller's order, 64 vertices a wave, and writing each
// source's 64 levels together (396 us). Levels of 255 and more are written to
// their place at once, and their bytes say so.
constexpr uint32_t kDeepLevel = 255;

__host__ __device__ constexpr uint32_t lev_row(uint32_t nsrc)
{
    uint32_t b = 4;  // at most 4 nsrc: the rows fit where nsrc rows of int32 do
    while (b < nsrc) b *= 2;
    return b;
}

// The four bytes of `x` that `bits` names become `b`'s.
__device__ __forceinline__ uint32_t put_bytes(uint32_t x, uint32_t bits, uint32_t b)
{
    const uint32_t m = (((bits & 15u) * 0x00204081u) & 0x01010101u) * 0xFFu;
    return (x & ~m) | (b & m);
}

// Byte `level` for the sources in `nw` into a vertex's row; `fresh`: none of
// its bytes counts yet.
__device__ __forceinline__ void put_levels(uint8_t *row, uint32_t bytes, uint64_t nw, bool fresh, uint32_t level)
{
    const uint32_t b = level * 0x01010101u;
    if (bytes < 16) {
        for (uint32_t d = 0; d < bytes / 4; d++) {
            uint32_t *x = (uint32_t *)row + d;
            const uint32_t bits = (uint32_t)(nw >> (4 * d)) & 15u;
            if (bits) *x = put_bytes(fresh ? 0u : *x, bits, b);
        }
        return;
    }
#pragma unroll
    for (uint32_t c = 0; c < 4; c++) {
        const uint32_t bits = (uint32_t)(nw >> (16 * c)) & 0xFFFFu;
        if (16 * c >= bytes || !bits) continue;
        uint4 x = make_uint4(0u, 0u, 0u, 0u);
        if (!fresh) x = ((uint4 *)row)[c];
        x.x = put_bytes(x.x, bits, b);
        x.y = put_bytes(x.y, bits >> 4, b);
        x.z = put_bytes(x.z, bits >> 8, b);
        x.w = put_bytes(x.w, bits >> 12, b);
        ((uint4 *)row)[c] = x;
    }
}

template <int BS>
__global__ __launch_bounds__(BS) void k_msbfs(MsBfsArgs a)
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
    const uint64_t bm = a.nsrc >= 64 ? ~0ull : ((1ull << a.nsrc) - 1);
    const uint32_t lb = lev_row(a.nsrc);

    __shared__ unsigned long long s_red[2][WPB];
    __shared__ unsigned long long s_lvl[5];
    __shared__ uint32_t s_len, s_at[WPB];

    for (uint32_t v = gtid; v < n; v += nthreads) {
        a.seen[v] = 0;
        a.F[v] = 0;
        a.F[(size_t)n + v] = 0;
        a.F[2 * (size_t)n + v] = 0;
    }
    if (blockIdx.x == 0) {
        clear_ctr(&a.ctr[0]);
        clear_ctr(&a.ctr[1]);
        clear_ctr(&a.ctr[2]);
        if (threadIdx.x == 0) {
            a.ctl[1] = 0;
            a.ctl[2] = 0;
            a.ctl[3] = 0;
        }
    }
    bool ok = grid_sync(a.bar, xcc, gen, a.abort);
    if (ok && blockIdx.x == 0 && threadIdx.x < kWave) {
        const bool has = (uint32_t)ln < a.nsrc;
        const uint32_t v = has ? a.src.get(ln) : 0u;
        uint64_t m = 0;
        int firstl = 64;
        for (int t = 0; t < 64; t++) {
            const uint32_t vt = lane_value(v, t);
            if (has && (uint32_t)t < a.nsrc && vt == v) {
                m |= 1ull << t;
                firstl = min(firstl, t);
            }
        }
        const bool lead = has && firstl == ln;
        if (has) {
            if (a.lev) a.lev[(size_t)v * lb + ln] = 0;
            else a.out[out_row(a.orow, ln, n) + v] = 0;
        }
        if (lead) {
            a.seen[v] = m;
            a.F[v] = m;
        }
        append_pair(&a.ctl[2], a.ring_v, a.ring_m, n, &a.ctl[1], lead, v, m);
        const uint32_t dv = lead ? g.row[v + 1] - g.row[v] : 0u;
        const unsigned long long sc = wave_sum_u64(dv);
        const unsigned long long cn = wave_sum_u64(lead ? 1ull : 0ull);
        if (ln == 0) {
            a.ctr[0].stripe[0].scout = sc;
            a.ctr[0].stripe[0].count = cn;
        }
    }
    if (ok) ok = grid_sync(a.bar, xcc, gen, a.abort);

    uint32_t L = 0, prev_len = 0;
    uint32_t pushes = 0, pulls = 0;
    unsigned long long ptrace = 0;
    DirectionPolicy pol{a.alpha, a.beta, (uint32_t)min(a.total_wl, 4294967295.0), n, a.force};
    while (ok) {
        read_counts(&a.ctr[L % 3], s_lvl);
        if (threadIdx.x == 0) s_len = __hip_atomic_load(&a.ctl[2 + (L & 1)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        const RoundCounts rc = unpack_counts(s_lvl, 0xFFFFFFFFu);
        const uint32_t len = min(s_len, n);
        __syncthreads();
        if (rc.count == 0 || (a.max_rounds && L >= a.max_rounds)) break;
        // the other half held level L-1, whose count every block read a level ago
        if (gtid == 0) a.ctl[2 + ((L + 1) & 1)] = 0;
        const bool pull = pol.next(L, rc.count, rc.scout);
        if (pull) {
            pulls++;
            if (L < 64) ptrace |= 1ull << L;
        } else {
            pushes++;
        }
        if (gtid == 0) write_trace(a.trace, L, pull, rc.count, rc.scout, t_start);
        if (blockIdx.x == 0) clear_ctr(&a.ctr[(L + 2) % 3]);
        const uint64_t *Fc = a.F + (size_t)(L % 3) * n;
        uint64_t *Fn = a.F + (size_t)((L + 1) % 3) * n;
        uint64_t *Ff = a.F + (size_t)((L + 2) % 3) * n;
        const size_t half = (size_t)(L & 1) * n, other = (size_t)((L + 1) & 1) * n;
        for (uint32_t i = gtid; i < prev_len; i += nthreads) Ff[a.ring_v[other + i]] = 0;

        ms_discover(g, a.seen, Fc, Fn, a.ring_v + half, a.ring_m + half, len, bm, pull, gwave, nwaves);
        ok = grid_sync(a.bar, xcc, gen, a.abort);
        if (!ok) break;

        unsigned long long scout = 0, cnt = 0;
        append_level<WPB>(Fn, n, W, gwave, nwaves, &a.ctl[2 + ((L + 1) & 1)], a.ring_v + other, a.ring_m + other, n,
                          &a.ctl[1], s_at);
        for (uint32_t w = gwave; w < W; w += nwaves) {
            const uint32_t v = w * 64 + ln;
            const uint64_t nw = v < n ? Fn[v] : 0ull;
            if (nw) {
                const uint64_t old = a.seen[v];
                a.seen[v] = old | nw;
                scout += g.row[v + 1] - g.row[v];
                cnt++;
                if (a.lev) put_levels(a.lev + (size_t)v * lb, lb, nw, old == 0, min(L + 1, kDeepLevel));
            }
            if (a.lev) {
                if (L + 1 >= kDeepLevel) {
                    uint64_t left = nw;
                    const uint32_t at = nw ? a.perm[v] : 0u;
                    while (left) {
                        const int s = first_lane(left);
                        left &= left - 1;
                        a.out[out_row(a.orow, s, n) + at] = (int32_t)(L + 1);
                    }
                }
                continue;
            }
            // one pass per source present in this word: lanes write consecutive vertices
            uint64_t any = wave_or_u64(nw);
            while (any) {
                const int s = __ffsll((unsigned long long)any) - 1;
                any &= any - 1;
                if ((nw >> s) & 1) a.out[out_row(a.orow, s, n) + v] = (int32_t)(L + 1);
            }
        }
        publish_counts<WPB>(&a.ctr[(L + 1) % 3], scout, cnt, false, s_red);
        pol.pull_prev = pull;
        prev_len = len;
        L++;
        ok = grid_sync(a.bar, xcc, gen, a.abort);
    }
    // -1 where no query of the batch came by (every block left the loop after
    // the same barrier, and `seen` holds all levels)
    if (ok && a.lev) {
        for (uint32_t w = gwave; w < W; w += nwaves) {
            const uint32_t v = w * 64 + ln;
            if (v >= n) break;
            const uint32_t u = a.inv[v];
            const uint64_t seen = a.seen[u];
            const uint8_t *row = a.lev + (size_t)u * lb;
            uint32_t x[16];
            if (lb < 16) {
                for (uint32_t d = 0; d < 4; d++) x[d] = d < lb / 4 && seen ? ((const uint32_t *)row)[d] : 0u;
            } else {
#pragma unroll
                for (uint32_t c = 0; c < 4; c++) {
                    uint4 y = make_uint4(0u, 0u, 0u, 0u);
                    if (16 * c < lb && seen) y = ((const uint4 *)row)[c];
                    x[4 * c] = y.x;
                    x[4 * c + 1] = y.y;
                    x[4 * c + 2] = y.z;
                    x[4 * c + 3] = y.w;
                }
            }
#pragma unroll
            for (uint32_t s = 0; s < 64; s++) {
                if (s >= a.nsrc) break;
                const uint32_t b = (x[s / 4] >> (8 * (s % 4))) & 0xFFu;
                const bool in = (seen >> s) & 1;
                // streamed past the L2, which the rows are being read through
                // (RMAT-19, 64 sources: 416 us by plain stores, 396 so)
                if (!in || b != kDeepLevel)
                    __builtin_nontemporal_store(in ? (int32_t)b : -1, &a.out[out_row(a.orow, s, n) + v]);
            }
        }
    } else if (ok)
        for (uint32_t w = gwave; w < W; w += nwaves) {
            const uint32_t v = w * 64 + ln;
            const uint64_t not_seen = v < n ? bm & ~a.seen[v] : 0ull;
            uint64_t any = wave_or_u64(not_seen);
            while (any) {
                const int s = first_lane(any);
                any &= any - 1;
                if ((not_seen >> s) & 1) a.out[out_row(a.orow, s, n) + v] = -1;
            }
        }
    if (gtid == 0) {
        DevStats s = a.first ? DevStats{} : *a.stats;
        s.rounds += L;
        s.push_rounds += pushes;
        s.pull_rounds += pulls;
        s.trace = ptrace;
        s.max_depth = max(s.max_depth, L ? L - 1 : 0u);
        s.iterations += 1;
        if (s.status == SG_OK) s.status = ok ? (a.ctl[1] ? SG_ERR_CAPACITY : SG_OK) : SG_ERR_TIMEOUT;
        *a.stats = s;
    }
    bar_end(a.bar);
}

// ----------------------------------------------------------- multi-source SSSP
// Up to 64 independent SSSP queries in one launch. Distances live as rows
// dist[v][2^qbits] (the batch rounded up to a power of two; lane q of a group
// of 2^qbits = query q), so an edge's end is one coalesced row for every
// query. A vertex's mask holds the queries that lowered its distance last
// round. A push round relaxes the out-edges of every vertex with a mask: a row
// read, an atomicMin per improving lane and one on the head's mask per edge; a
// vertex enters the next round's entry list when the first bit of its next
// mask is set (the atomicOr returns 0). A pull round has every vertex take the
// minimum over its in-edges from vertices with a mask, its row in registers:
// no atomics but for in-hubs split into chunks. Results leave
// transposed, one contiguous n-vector per query in the order asked for, equal
// to sg_sssp from that source.
struct MsSsspArgs {
    DevGraph g;
    MsSources src;
    uint32_t first;       // start the summary (else: add to it)
    uint32_t nsrc;
    uint32_t *dist;       // [n][2^qbits]
    uint64_t *F;          // 3 x n masks, round r in F + (r % 3) n
    uint32_t *out;        // distances of source q in row out_row(orow, q)
    const uint32_t *orow;
    const uint32_t *inv;  // out[v] is device vertex inv[v]'s (null: v's)
    int32_t force;        // 0: push rounds only
    uint32_t *ring;       // 3 x n: entries of round r in third r % 3
    uint32_t *cmin;       // 3 x 64: smallest distance queued for round r by each
                          // query, complemented (0: none), in third r % 3
    FrontierCtr *ctr;     // 3 slots: entries / out-degree of each round
    GridBarrier bar;
    uint32_t *abort;
    DevStats *stats;
    DevTrace *trace;
    uint32_t max_rounds;
    uint32_t probe;
};

struct MsRelax {
    const MsSsspArgs *a;
    uint64_t *Fn;
    Stager S;        // the next round's entries
    uint32_t qbits;  // queries of the batch fit in 2^qbits lanes
    unsigned long long scout, count;
    uint32_t fmin;   // this lane's query has no frontier distance below this
    uint32_t minv;   // smallest distance this lane queued for the next round
};

// Edge steps a group of lanes keeps in flight in the batched relaxation.
#ifndef SG_MS_RELAX_STEPS
#define SG_MS_RELAX_STEPS 16
#endif
constexpr int kMsRelaxSteps = SG_MS_RELAX_STEPS;

// Relax the out-edges [b, e) of u for the queries in `mask`. The wave is
// split into 64 / 2^qbits groups; each group takes kMsRelaxSteps edges per
// step, with the loads and atomics of all of them issued before any result is
// used, so a batch of B queries keeps about 64 / B x kMsRelaxSteps edges in
// flight per wave. A group's leader publishes the queries whose distance it
// lowered into the next round's mask of the edge's head; the heads whose mask
// it was first to set are staged for the next round's entries.
__device__ __forceinline__ void ms_relax_range(MsRelax &R, uint32_t u, uint32_t b, uint32_t e, uint64_t mask)
{
    constexpr int U = kMsRelaxSteps;
    const MsSsspArgs &a = *R.a;
    const DevGraph &g = a.g;
    const int ln = lane();
    const uint32_t qb = R.qbits;
    const uint32_t q = (uint32_t)ln & ((1u << qb) - 1), grp = (uint32_t)ln >> qb, ngrp = 64u >> qb;
    const uint64_t gmask = qb == 6 ? ~0ull : ((1ull << (1u << qb)) - 1);
    const bool mine = (mask >> q) & 1;
    const uint32_t du = mine ? a.dist[((size_t)u << qb) + q] : 0xFFFFFFFFu;
    for (uint32_t e0 = b; e0 < e; e0 += ngrp * U) {
        uint32_t v[U], nd[U], cur[U];
        bool act[U];
#pragma unroll
        for (int s = 0; s < U; s++) {
            const uint32_t ed = e0 + grp + (uint32_t)s * ngrp;
            act[s] = ed < e;
            v[s] = act[s] ? g.col[ed] : 0u;
            const uint32_t w = (act[s] && mine) ? (g.w ? g.w[ed] : 1u) : 0u;
            nd[s] = du > 0xFFFFFFFFu - w ? 0xFFFFFFFFu : du + w;
            act[s] = act[s] && mine;
        }
#pragma unroll
        for (int s = 0; s < U; s++) cur[s] = act[s] ? a.dist[((size_t)v[s] << qb) + q] : 0u;
        // every atomic of the step is issued before any result is read (a
        // result consumed inside its own branch makes each one wait in turn)
        uint32_t old[U];
#pragma unroll
        for (int s = 0; s < U; s++) {
            old[s] = 0xFFFFFFFFu;
            if (act[s] && nd[s] < cur[s]) old[s] = atomicMin(&a.dist[((size_t)v[s] << qb) + q], nd[s]);
        }
        unsigned long long fo[U];
#pragma unroll
        for (int s = 0; s < U; s++) {
            const bool imp = act[s] && nd[s] < cur[s] && nd[s] < old[s];
            if (imp) R.minv = min(R.minv, nd[s]);
            const uint64_t im = ballot(imp);
            const uint64_t gm = (im >> (grp << qb)) & gmask;
            fo[s] = ~0ull;
            if (q == 0 && gm) fo[s] = atomicOr((unsigned long long *)&R.Fn[v[s]], (unsigned long long)gm);
        }
        // heads whose mask this wave set first, staged in the block's LDS: an
        // append per wave and step to one global counter had serialised at
        // 11 ns each (131 K entries: 580 us a round)
#pragma unroll
        for (int s = 0; s < U; s++) {
            const bool fresh = fo[s] == 0;
            if (fresh) {
                R.scout += g.row[v[s] + 1] - g.row[v[s]];
                R.count++;
            }
            stage(R.S, fresh, v[s]);
        }
    }
}

// Rows a group keeps in flight in a pull round.
constexpr int kMsPullRows = 8;
// A round pulls when its entries' out-edges number at least 1/kMsPullRatio of
// all edges, and when the batch fills groups of at least 2^kMsPullBits lanes: a
// pull round reads every vertex's in-edges, but a row only where it can still
// lower something, and without atomics. 24 queries on 230 017 vertices, 3.4 M
// edges: 500 us a dense round by pushing, 250 falling to 180 by pulling; whole
// call 3180 us without pull rounds, 1759 with a ratio of 4, 1621 with 16, 1569
// with 32 (64: 1541, but a 150 x 200 grid loses what that gains). Narrow groups walk too
// few edges at a time: 8 queries on 60 001 vertices take 602 us pushing and 702
// pulling, 16 take 859 and 703. Groups of 16 lanes walk an in-hub's chunk in 16 steps,
// which a graph of few vertices has too little other work to hide: with in-hubs they
// pull from kMsPullNarrow vertices on (16 queries on R-MAT graphs: 4096 vertices, 97 K
// edges 607 us pulling and 428 pushing, 8192, 111 K 569 and 487, 16 384, 120 K 638 and 749;
// without in-hubs, 8000 vertices of mean degree 15: 300 and 365).
#ifndef SG_MS_PULL_RATIO
#define SG_MS_PULL_RATIO 32
#endif
constexpr uint32_t kMsPullRatio = SG_MS_PULL_RATIO;
#ifndef SG_MS_PULL_BITS
#define SG_MS_PULL_BITS 4
#endif
constexpr uint32_t kMsPullBits = SG_MS_PULL_BITS;
constexpr uint32_t kMsPullNarrow = 12288;

// In-edges a group is about to read the far ends of: one per lane.
struct MsEdges {
    uint32_t u, w;
    bool in;
};

__device__ __forceinline__ MsEdges ms_edges(const DevGraph &g, uint32_t ed, uint32_t e)
{
    MsEdges x{0u, 0u, ed < e};
    if (x.in) {
        x.u = g.csrc[ed];
        x.w = g.cw ? g.cw[ed] : 1u;
    }
    return x;
}

// Smallest candidate below `best` of this lane's query over the edges `x` from
// vertices with a mask in Fc, or `best`. A row is read by the lanes whose query
// the edge can still improve (every frontier distance is at least fmin).
// Wave-convergent.
__device__ __forceinline__ uint32_t ms_pull_edges(const MsRelax &R, const uint64_t *Fc, const MsEdges &x, uint32_t best)
{
    const MsSsspArgs &a = *R.a;
    const int ln = lane();
    const uint32_t qb = R.qbits, width = 1u << qb;
    const uint32_t q = (uint32_t)ln & (width - 1);
    const int base = ln & ~(int)(width - 1);  // the group's first lane
    const uint64_t gmask = qb == 6 ? ~0ull : ((1ull << width) - 1);
    const uint64_t f = x.in ? Fc[x.u] : 0ull;
    uint64_t live = (ballot(f != 0) >> base) & gmask;  // the group's edges to read
    while (ballot(live != 0)) {
        uint32_t d[kMsPullRows], wt[kMsPullRows];
#pragma unroll
        for (int k = 0; k < kMsPullRows; k++) {
            const bool on = live != 0;
            const int j = base + (on ? first_lane(live) : 0);
            live &= live - 1;
            const uint32_t uj = shfl(x.u, j);
            const uint64_t fj = shfl(f, j);
            wt[k] = shfl(x.w, j);
            const bool can = on && ((fj >> q) & 1) && (uint64_t)R.fmin + wt[k] < best;
            d[k] = can ? a.dist[((size_t)uj << qb) + q] : 0xFFFFFFFFu;
        }
#pragma unroll
        for (int k = 0; k < kMsPullRows; k++) best = min(best, d[k] > 0xFFFFFFFFu - wt[k] ? 0xFFFFFFFFu : d[k] + wt[k]);
    }
    return best;
}

// A pull round: in-hubs by the chunk list, a chunk per group merged with
// atomicMin, then every other vertex, a group each. Either way a group stops at
// once where no query of it can be lowered (see sssp_dev.hpp's settled()).
__device__ __forceinline__ void ms_pull(MsRelax &R, const uint64_t *Fc, uint32_t nsrc, uint32_t gwave, uint32_t nwaves)
{
    const MsSsspArgs &a = *R.a;
    const DevGraph &g = a.g;
    const int ln = lane();
    const uint32_t qb = R.qbits, width = 1u << qb, ngrp = 64u >> qb;
    const uint32_t q = (uint32_t)ln & (width - 1), grp = (uint32_t)ln >> qb;
    const uint64_t gmask = qb == 6 ? ~0ull : ((1ull << width) - 1);
    const bool has = q < nsrc;
    // whether some query of the group can be lowered below its d
    auto open = [&](uint32_t d, uint32_t mw) {
        return ((ballot(has && (uint64_t)R.fmin + mw < d) >> (grp << qb)) & gmask) != 0;
    };
    // the group's lowered queries into v's next mask, v into the next entries
    auto publish = [&](bool low, uint32_t v, uint32_t d, bool shared) {
        if (low) R.minv = min(R.minv, d);
        const uint64_t bits = (ballot(low) >> (grp << qb)) & gmask;
        bool fresh = false;
        if (q == 0 && bits) {
            if (shared) {
                fresh = atomicOr((unsigned long long *)&R.Fn[v], (unsigned long long)bits) == 0;
            } else {
                R.Fn[v] = bits;
                fresh = true;
            }
        }
        if (fresh) {
            R.scout += g.row[v + 1] - g.row[v];
            R.count++;
        }
        stage(R.S, fresh, v);
    };
    const uint32_t step = nwaves * ngrp;
    for (uint32_t c0 = gwave * ngrp; c0 < g.nhugein; c0 += step) {
        const uint32_t c = c0 + grp;
        uint32_t v = 0, b = 0, e = 0, d0 = 0, mw = 0;
        if (c < g.nhugein) {
            const uint2 dsc = g.hugein[c];
            v = dsc.x;
            b = dsc.y;
            e = min(g.cstart[v + 1], b + kPullChunk);
            d0 = a.dist[((size_t)v << qb) + q];
            mw = g.cminw ? g.cminw[v] : (g.cw ? 0u : 1u);
        }
        if (!open(d0, mw)) e = b;
        uint32_t best = d0;
        MsEdges x = ms_edges(g, b + q, e);
        for (; ballot(b < e); b += width) {
            const MsEdges y = ms_edges(g, b + width + q, e);  // the next ones, while these are worked
            best = ms_pull_edges(R, Fc, x, best);
            x = y;
        }
        bool low = has && best < d0;
        if (low) low = best < atomicMin(&a.dist[((size_t)v << qb) + q], best);
        publish(low, v, best, true);
    }
    // Every other vertex: the next one's row, first edges and smallest weight are
    // read while this one is worked, the edge range of the one after it too.
    auto range = [&](uint32_t v, uint32_t &b, uint32_t &e) {
        b = e = 0;
        if (v < g.n) {
            b = g.cstart[v];
            e = g.cstart[v + 1];
            if (e - b > kPullHubDegree) e = b;
        }
    };
    auto head = [&](uint32_t v, uint32_t b, uint32_t e, uint32_t &d, uint32_t &mw, MsEdges &x) {
        d = mw = 0;
        x = ms_edges(g, b + q, e);
        if (b < e) {
            d = a.dist[((size_t)v << qb) + q];
            mw = g.cminw ? g.cminw[v] : (g.cw ? 0u : 1u);
        }
    };
    uint32_t v = gwave * ngrp + grp, b, e, b1, e1, d0, mw;
    MsEdges x;
    range(v, b, e);
    range(v + step, b1, e1);
    head(v, b, e, d0, mw, x);
    for (uint32_t v0 = gwave * ngrp; v0 < g.n; v0 += step, v += step) {
        uint32_t b2, e2, d1, mw1;
        MsEdges x1;
        range(v + 2 * step, b2, e2);
        head(v + step, b1, e1, d1, mw1, x1);
        if (!open(d0, mw)) {
            e = b;
            x.in = false;
        }
        uint32_t best = d0;
        for (; ballot(b < e); b += width) {
            best = ms_pull_edges(R, Fc, x, best);
            x = ms_edges(g, b + width + q, e);
        }
        const bool low = has && best < d0;
        if (ballot(low)) {
            if (low) a.dist[((size_t)v << qb) + q] = best;
            publish(low, v, best, false);
        }
        b = b1;
        e = e1;
        b1 = b2;
        e1 = e2;
        d0 = d1;
        mw = mw1;
        x = x1;
    }
}

template <int BS>
__global__ __launch_bounds__(BS) void k_mssssp(MsSsspArgs a)
{
    if (a.probe) {
        residency_probe(a.bar.words, 1u << 20);
        return;
    }
    constexpr int WPB = BS / kWave;
    const DevGraph &g = a.g;
    const uint32_t n = g.n;
    const uint32_t gtid = blockIdx.x * BS + threadIdx.x;
    const uint32_t nthreads = gridDim.x * BS;
    const uint32_t gwave = blockIdx.x * WPB + threadIdx.x / kWave;
    const uint32_t nwaves = gridDim.x * WPB;
    const int ln = lane();
    const uint32_t xcc = xcc_id();
    BarState gen = bar_begin(a.bar, xcc);
    const long long t_start = wall_clock64();
    uint32_t qbits = 0;
    while ((1u << qbits) < a.nsrc) qbits++;

    __shared__ unsigned long long s_red[2][WPB];
    __shared__ unsigned long long s_lvl[5];
    constexpr uint32_t kLdsQ = 8u * BS;
    __shared__ uint32_t s_q[kLdsQ];
    __shared__ uint32_t s_qn, s_flush[2], s_min[64];

    for (size_t i = gtid; i < (size_t)n << qbits; i += nthreads) a.dist[i] = 0xFFFFFFFFu;
    for (size_t i = gtid; i < 3 * (size_t)n; i += nthreads) a.F[i] = 0;
    if (blockIdx.x == 0) {
        clear_ctr(&a.ctr[0]);
        clear_ctr(&a.ctr[1]);
        clear_ctr(&a.ctr[2]);
        if (threadIdx.x < 3 * 64) a.cmin[threadIdx.x] = threadIdx.x < 64 ? ~0u : 0u;  // round 0: distance 0
    }
    bool ok = grid_sync(a.bar, xcc, gen, a.abort);
    if (ok && blockIdx.x == 0 && threadIdx.x < kWave) {
        const bool has = (uint32_t)ln < a.nsrc;
        const uint32_t v = has ? a.src.get(ln) : 0u;
        uint64_t m = 0;
        int firstl = 64;
        for (int t = 0; t < 64; t++) {
            const uint32_t vt = lane_value(v, t);
            if (has && (uint32_t)t < a.nsrc && vt == v) {
                m |= 1ull << t;
                firstl = min(firstl, t);
            }
        }
        const bool lead = has && firstl == ln;
        if (has) a.dist[((size_t)v << qbits) + ln] = 0;
        if (lead) a.F[v] = m;
        const uint64_t lm = ballot(lead);
        if (lead) a.ring[rank_in(lm)] = v;
        const uint32_t dv = lead ? g.row[v + 1] - g.row[v] : 0u;
        const unsigned long long sc = wave_sum_u64(dv);
        if (ln == 0) {
            a.ctr[0].qlen = (uint32_t)__popcll(lm);
            a.ctr[0].stripe[0].scout = sc;
            a.ctr[0].stripe[0].count = (unsigned long long)__popcll(lm);
        }
    }
    if (ok) ok = grid_sync(a.bar, xcc, gen, a.abort);

    const bool pullable =
        qbits > kMsPullBits || (qbits == kMsPullBits && (n >= kMsPullNarrow || g.nhugein == 0));
    uint32_t r = 0, prev_len = 0, pulls = 0;
    unsigned long long ptrace = 0;
    while (ok) {
        read_counts(&a.ctr[r % 3], s_lvl);
        if (threadIdx.x == 0) s_qn = 0;
        __syncthreads();
        const RoundCounts rc = unpack_counts(s_lvl, n);
        const uint32_t len = rc.qlen;
        __syncthreads();
        if (rc.count == 0 || (a.max_rounds && r >= a.max_rounds)) break;
        const bool pull = a.force != 0 && pullable && rc.scout * kMsPullRatio >= g.m;
        pulls += pull;
        if (pull && r < 64) ptrace |= 1ull << r;
        if (gtid == 0) write_trace(a.trace, r, pull, rc.count, rc.scout, t_start);
        if (blockIdx.x == 0) {
            clear_ctr(&a.ctr[(r + 2) % 3]);
            if (threadIdx.x < 64) a.cmin[(r + 2) % 3 * 64 + threadIdx.x] = 0;
        }
        if (threadIdx.x < 64) s_min[threadIdx.x] = 0xFFFFFFFFu;  // (a barrier of the round's end orders this)
        const uint64_t *Fc = a.F + (size_t)(r % 3) * n;
        uint64_t *Ff = a.F + (size_t)((r + 2) % 3) * n;
        const uint32_t *cur = a.ring + (size_t)(r % 3) * n;
        const uint32_t *old = a.ring + (size_t)((r + 2) % 3) * n;
        for (uint32_t i = gtid; i < prev_len; i += nthreads) Ff[old[i]] = 0;

        // (a vertex enters a round's entries once, so n entries hold them all)
        MsRelax R{&a, a.F + (size_t)((r + 1) % 3) * n,
                  Stager{a.ring + (size_t)((r + 1) % 3) * n, n, &a.ctr[(r + 1) % 3], s_q, &s_qn, kLdsQ}, qbits, 0, 0, 0, 0xFFFFFFFFu};
        const uint32_t q = (uint32_t)ln & ((1u << qbits) - 1);
        R.fmin = ~__hip_atomic_load(&a.cmin[r % 3 * 64 + q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (pull) ms_pull(R, Fc, a.nsrc, gwave, nwaves);
        // hubs through the static chunk list
        for (uint32_t c = gwave; !pull && c < g.nhuge; c += nwaves) {
            const uint2 dsc = g.huge[c];
            const uint64_t mk = Fc[dsc.x];
            if (mk) ms_relax_range(R, dsc.x, dsc.y, min(g.row[dsc.x + 1], dsc.y + kHugeChunk), mk);
        }
        // (the entry after next, and the next one's edge range and mask, are
        // read while this one is relaxed)
        uint32_t i = pull ? len : gwave;
        uint32_t u1 = i < len ? cur[i] : 0u, u2 = i + nwaves < len ? cur[i + nwaves] : 0u;
        uint32_t b1 = g.row[u1], e1 = g.row[u1 + 1];
        uint64_t m1 = Fc[u1];
        for (; i < len; i += nwaves) {
            const uint32_t u = u1, b = b1, e = e1;
            const uint64_t mk = m1;
            u1 = u2;
            u2 = i + 2 * nwaves < len ? cur[i + 2 * nwaves] : 0u;
            b1 = g.row[u1];
            e1 = g.row[u1 + 1];
            m1 = Fc[u1];
            if (e - b > kHugeDegree) continue;
            ms_relax_range(R, u, b, e, mk);
        }
        publish_counts<WPB>(&a.ctr[(r + 1) % 3], R.scout, R.count, false, s_red);
        if (R.minv != 0xFFFFFFFFu) atomicMin(&s_min[q], R.minv);
        flush_stage(R.S, s_flush);
        if (threadIdx.x < 64 && s_min[threadIdx.x] != 0xFFFFFFFFu)
            atomicMax(&a.cmin[(r + 1) % 3 * 64 + threadIdx.x], ~s_min[threadIdx.x]);
        prev_len = len;
        r++;
        ok = grid_sync(a.bar, xcc, gen, a.abort);
    }
    // results, one contiguous row per query: tiles of 64 vertices go through
    // the block's LDS, rows read and written whole (the caller's order is a
    // permutation of rows here, and costs no pass of its own)
    if (ok) {
        static_assert(kLdsQ >= 64 * 9, "a tile of eight queries fits");
        constexpr uint32_t kTileQ = kLdsQ / 64 - 1 < 64 ? kLdsQ / 64 - 1 : 64;  // queries a tile holds
        const uint32_t qn = 1u << qbits;
        for (uint32_t v0 = blockIdx.x * 64; v0 < n; v0 += gridDim.x * 64) {
            for (uint32_t q0 = 0; q0 < a.nsrc; q0 += kTileQ) {
                const uint32_t qc = min(kTileQ, a.nsrc - q0);
                __syncthreads();
                for (uint32_t i = threadIdx.x; i < 64 * qn; i += BS) {
                    const uint32_t v = v0 + (i >> qbits), q = i & (qn - 1);
                    if (v < n && q - q0 < qc)
                        s_q[(q - q0) * 65 + (i >> qbits)] = a.dist[((size_t)(a.inv ? a.inv[v] : v) << qbits) + q];
                }
                __syncthreads();
                for (uint32_t i = threadIdx.x; i < 64 * qc; i += BS) {
                    const uint32_t v = v0 + (i & 63), q = i >> 6;
                    if (v < n) a.out[out_row(a.orow, q0 + q, n) + v] = s_q[q * 65 + (i & 63)];
                }
            }
        }
    }
    if (gtid == 0) {
        DevStats s = a.first ? DevStats{} : *a.stats;
        s.rounds += r;
        s.push_rounds += r - pulls;
        s.pull_rounds += pulls;
        s.trace = ptrace;
        s.max_depth = max(s.max_depth, r);
        s.iterations += 1;
        if (s.status == SG_OK) s.status = ok ? SG_OK : SG_ERR_TIMEOUT;
        *a.stats = s;
    }
    bar_end(a.bar);
}

}  // namespace


// ------------------------------------------------------------------ host side

namespace {

constexpr uint64_t al256(uint64_t x) { return (x + 255) / 256 * 256; }

// Offsets of each batched kind's working arrays inside the engine's arena.
struct MsLayout {
    uint64_t off[10];
    uint64_t total;
};

MsLayout ms_layout(int kind, uint64_t n)
{
    MsLayout L{};
    uint64_t o = 0;
    auto put = [&](int i, uint64_t bytes) {
        L.off[i] = o;
        o += al256(bytes);
    };
    if (kind == kMsBfs) {
        put(0, n * 8);      // seen
        put(1, 3 * n * 8);  // F
        put(2, 2 * n * 4);  // ring_v
        put(3, 2 * n * 8);  // ring_m
        put(4, 256);        // ctl
    } else if (kind == kMsSssp) {
        put(0, n * 64 * 4); // dist rows
        put(1, 3 * n * 8);  // F
        put(2, 3 * n * 4);  // ring
        put(4, 3 * 64 * 4); // cmin
    } else {
        const uint64_t cap = std::min<uint64_t>(n * 64 + 4096, 0xFFFFFFF0ull);
        put(0, n * 8);                             // seen
        put(1, 3 * n * 8);                         // F
        put(2, n * 64 * 8);                        // sigma
        put(3, n * 64 * 8);                        // psi
        put(5, n * 8);                             // bc accumulator
        put(6, cap * 4);                           // stack vertices
        put(7, cap * 8);                           // stack masks
        put(8, (uint64_t)(kMaxLevels + 4) * 4);    // level starts
        put(4, 256);                               // ctl
        L.off[9] = cap;
    }
    L.total = o;
    return L;
}

template <typename Args>
void fill_common(sg_engine *e, Args &a)
{
    a.g = e->g->dev;
    a.ctr = (FrontierCtr *)e->ctr;
    a.bar.spin_limit = 1u << 22;
    a.abort = e->abort_flag;
    a.stats = e->stats;
    a.trace = e->trace;
}

template <typename Args>
int launch_grid(sg_engine *e, const void *fn, int bs, Args &a)
{
    sg_engine::PGrid *pg = nullptr;
    auto probe = [e, a, fn, bs](int blocks, uint32_t *words) -> int {
        Args p = a;
        p.probe = 1;
        p.bar.words = words;
        void *params[] = {&p};
        SG_HIP(hipLaunchKernel(fn, dim3(blocks), dim3(bs), params, 0, e->stream));
        return SG_OK;
    };
    int rc = engine_persistent_grid(e, fn, bs, probe, &pg);
    if (rc) return rc;
    bind_barrier(pg, a.bar);
    return engine_launch_persistent(e, [&]() -> int {
        void *params[] = {&a};
        SG_HIP(hipLaunchKernel(fn, dim3(pg->blocks), dim3(bs), params, 0, e->stream));
        pg->launches++;
        return SG_OK;
    });
}

}  // namespace

namespace sg {

int ms_prepare(sg_engine *e, int kind)
{
    int rc = engine_ensure_bfs_state(e);
    if (rc) return rc;
    return engine_ensure_aux(e, ms_layout(kind, e->g->dev.n).total);
}

int ms_launch(sg_engine *e, int kind, const uint32_t *dev_src, uint32_t nsrc, void *out, const uint32_t *dev_orow,
              bool first, bool last, const uint32_t *inv, const uint32_t *host_src)
{
    if (nsrc < 1 || nsrc > 64) SG_FAIL(SG_ERR_RANGE, "batched launch: 1..64 sources");
    const uint64_t n = e->g->dev.n;
    const MsLayout L = ms_layout(kind, n);
    if (!e->aux || e->aux_bytes < L.total) SG_FAIL(SG_ERR_STATE, "batched launch: arena not prepared");
    char *base = (char *)e->aux;
    const sg_engine_options &o = e->opt;
    const int force = forced_direction(o);
    if (force < -1) SG_FAIL(SG_ERR_UNSUPPORTED, "batched launch: only data-driven push/pull variants apply");
    if (o.lb_push == SG_LB_NONE || o.lb_pull == SG_LB_NONE)
        SG_FAIL(SG_ERR_UNSUPPORTED, "batched launch: LoadBalancing::NONE applies to sg_bfs and sg_sssp only");
    const int bs = o.block_size ? o.block_size : 1024;
    if (bs != 256 && bs != 512 && bs != 1024) SG_FAIL(SG_ERR_UNSUPPORTED, "batched launch: block_size must be 256, 512 or 1024");
    const double alpha = o.alpha == 0.0 ? 1.0 : o.alpha;
    const double total_wl = (double)e->g->dev.m * o.edge_factor;
    MsSources src{};
    src.dev = dev_src;
    if (!dev_src) std::copy(host_src, host_src + nsrc, src.v);
    if (kind == kMsBfs) {
        MsBfsArgs a{};
        fill_common(e, a);
        a.src = src;
        a.first = first;
        a.nsrc = nsrc;
        a.seen = (uint64_t *)(base + L.off[0]);
        a.F = (uint64_t *)(base + L.off[1]);
        a.ring_v = (uint32_t *)(base + L.off[2]);
        a.ring_m = (uint64_t *)(base + L.off[3]);
        a.ctl = (uint32_t *)(base + L.off[4]);
        a.out = (int32_t *)out;
        a.orow = dev_orow;
        if (inv) {
            a.lev = (uint8_t *)e->work;
            a.inv = inv;
            a.perm = e->g->d_perm;
        }
        a.alpha = alpha;
        a.beta = o.beta;
        a.total_wl = total_wl;
        a.force = force;
        a.max_rounds = (uint32_t)o.max_iteration;
        const void *fn = bs == 256 ? (const void *)k_msbfs<256> : bs == 512 ? (const void *)k_msbfs<512> : (const void *)k_msbfs<1024>;
        return launch_grid(e, fn, bs, a);
    }
    if (kind == kMsSssp) {
        MsSsspArgs a{};
        fill_common(e, a);
        a.src = src;
        a.first = first;
        a.nsrc = nsrc;
        a.dist = (uint32_t *)(base + L.off[0]);
        a.F = (uint64_t *)(base + L.off[1]);
        a.ring = (uint32_t *)(base + L.off[2]);
        a.out = (uint32_t *)out;
        a.orow = dev_orow;
        a.inv = inv;
        a.cmin = (uint32_t *)(base + L.off[4]);
        a.force = force;
        a.max_rounds = (uint32_t)o.max_iteration;
        const void *fn = bs == 256 ? (const void *)k_mssssp<256> : bs == 512 ? (const void *)k_mssssp<512> : (const void *)k_mssssp<1024>;
        return launch_grid(e, fn, bs, a);
    }
    BcArgs a{};
    fill_common(e, a);
    a.src = src;
    a.nsrc = nsrc;
    a.seen = (uint64_t *)(base + L.off[0]);
    a.F = (uint64_t *)(base + L.off[1]);
    a.sigma = (double *)(base + L.off[2]);
    a.psi = (double *)(base + L.off[3]);
    a.bc = (double *)(base + L.off[5]);
    a.stk_v = (uint32_t *)(base + L.off[6]);
    a.stk_m = (uint64_t *)(base + L.off[7]);
    a.lvl = (uint32_t *)(base + L.off[8]);
    a.cap = (uint32_t)L.off[9];
    a.ctl = (uint32_t *)(base + L.off[4]);
    if (kind == kMsBcDep) {
        a.dep = (float *)out;
        a.orow = dev_orow;
        a.out = nullptr;
        a.last = 0;
    } else {
        a.out = (float *)out;
        a.last = last;
    }
    a.first = first;
    a.alpha = alpha;
    a.beta = o.beta;
    a.total_wl = total_wl;
    a.force = force;
    const void *fn = bs == 256 ? (const void *)k_bc<256> : bs == 512 ? (const void *)k_bc<512> : (const void *)k_bc<1024>;
    return launch_grid(e, fn, bs, a);
}

}  // namespace sg

namespace {

// C-ABI driver: k host sources in batches of `batch`, results in the value
// array (row i for sources[i], or the BC sum).
int ms_run(sg_engine *e, int kind, const uint32_t *sources, int32_t k, int32_t batch, const char *name)
{
    if (!e || !sources) SG_FAIL(SG_ERR_INVALID, std::string(name) + ": null argument");
    if (k < 1) SG_FAIL(SG_ERR_RANGE, std::string(name) + ": need at least one source");
    if (batch == 0) batch = 64;
    if (batch < 1 || batch > 64) SG_FAIL(SG_ERR_RANGE, std::string(name) + ": batch must be in [1, 64]");
    const DevGraph &d = e->g->dev;
    for (int32_t i = 0; i < k; i++)
        if (sources[i] >= d.n) SG_FAIL(SG_ERR_RANGE, std::string(name) + ": source >= n");
    if (forced_direction(e->opt) < -1)
        SG_FAIL(SG_ERR_UNSUPPORTED, std::string(name) + ": only data-driven push/pull variants apply");
    if (e->opt.lb_push == SG_LB_NONE || e->opt.lb_pull == SG_LB_NONE)
        SG_FAIL(SG_ERR_UNSUPPORTED, std::string(name) + ": LoadBalancing::NONE applies to sg_bfs and sg_sssp only");
    const bool single_bc = batch == 1 && (kind == kMsBcDep || kind == kMsBcSum);
    int rc = single_bc ? engine_ensure_bfs_state(e) : ms_prepare(e, kind);
    if (rc) return rc;
    const uint64_t n = d.n;
    const uint64_t rows = kind == kMsBcSum ? 1 : (uint64_t)k;
    void *res = nullptr;
    // batched BFS and SSSP write the caller's order themselves
    const bool direct = kind == kMsSssp || kind == kMsBfs;
    if (kind == kMsBfs) {
        // (a relabelled graph's level rows are kept in the work rows)
        if ((rc = engine_result_rows(e, rows, &res))) return rc;
        res = e->value;
    } else if (direct) {
        if ((rc = engine_ensure_value(e, rows * n * 4))) return rc;
        res = e->value;
    } else if ((rc = engine_result_rows(e, rows, &res))) {
        return rc;
    }
    // (the kernels' arguments carry the sources: nothing is left to wait for)
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    SG_HIP(hipStreamIsCapturing(e->stream, &cap));
    if (cap != hipStreamCaptureStatusNone) SG_FAIL(SG_ERR_HIP, std::string(name) + ": not on a capturing stream");
    std::vector<uint32_t> dsrc(k);
    for (int32_t i = 0; i < k; i++) dsrc[i] = dev_vertex(e->g, sources[i]);
    e->last_algo = 3 + kind;
    // one source per launch (the single-source kernel, no bit-packed rows), or
    // a batch. A single launch's time is the device's clock, several take events.
    const int per = single_bc ? 1 : batch, nb = (k + per - 1) / per;
    if (nb > 1) SG_HIP(hipEventRecord(e->ev0, e->stream));
    for (int i = 0; i < nb; i++) {
        const bool first = i == 0, last = i == nb - 1;
        if (single_bc) {
            float *dep = kind == kMsBcDep ? (float *)res + (size_t)i * n : nullptr;
            float *sum = kind == kMsBcSum ? (float *)res : nullptr;
            rc = bc1_launch(e, dsrc[i], dep, nullptr, sum, first, last);
        } else {
            const uint32_t ns = (uint32_t)std::min(batch, k - i * batch);
            void *out = kind == kMsBcSum ? res : (void *)((uint32_t *)res + (size_t)i * batch * n);
            rc = ms_launch(e, kind, nullptr, ns, out, nullptr, first, last,
                           direct && e->g->relabeled ? e->g->d_inv : nullptr, dsrc.data() + (size_t)i * batch);
        }
        if (rc) return rc;
    }
    if (nb > 1) SG_HIP(hipEventRecord(e->ev1, e->stream));
    if (!direct && (rc = engine_finish(e, rows))) return rc;
    e->timed = true;
    e->clocked = nb > 1 ? nullptr : e->last_grid;
    return SG_OK;
}

}  // namespace

extern "C" int sg_bc(sg_engine *e, const uint32_t *sources, int32_t k, int32_t batch)
{
    return ms_run(e, kMsBcSum, sources, k, batch, "sg_bc");
}

extern "C" int sg_bc_dependency(sg_engine *e, const uint32_t *sources, int32_t k, int32_t batch)
{
    return ms_run(e, kMsBcDep, sources, k, batch, "sg_bc_dependency");
}

extern "C" int sg_bfs_multi(sg_engine *e, const uint32_t *sources, int32_t k, int32_t batch)
{
    return ms_run(e, kMsBfs, sources, k, batch, "sg_bfs_multi");
}

extern "C" int sg_sssp_multi(sg_engine *e, const uint32_t *sources, int32_t k, int32_t batch)
{
    return ms_run(e, kMsSssp, sources, k, batch, "sg_sssp_multi");
}
