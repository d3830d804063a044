// kNN and radius search with one wavefront per query, for gfx950 (k or cap <=
// kWaveMaxK; a radius search is a kNN search of its cap with a limit).
//
// A wave takes up to 64 consecutive queries of the cell-sorted order, one at
// a time.  The 3x3x3 cells around a query's cell, on the finest pyramid level
// where they hold enough points, are its region; their points are loaded once
// for all queries of the cell and stay in registers, up to 12 per lane.  For
// each query the lanes compute the distances of their points and a threshold
// that leaves between k and 16 G of them is found by counting (ballots).  The
// kept candidates go to LDS; when 64 / G queries are collected, G lanes sort
// the row of each in registers and the wave writes the rows.  A query whose
// threshold reaches past its region scans the cells of that ball; one whose
// region holds too few points (or too many for the registers) scans balls that
// grow until they hold k.  The fused mode ends with the features, one query
// per lane.
//
// What bounds it: instruction issue and the latency of the few dependent
// loads per region, at 12 or 13 waves per CU (registers; LDS rows):
// 10 M LiDAR points at k = 20 take about 200 vector instructions per query
// (k_search, a lane per query with a heap, about 430, its lanes waiting for
// each other: 3 times the candidate steps and 3.5 times the insertions of a
// lane).  Search kernels per call, k_search -> this one: 10 M at k = 20 9.8 ->
// 5.9 ms, 4 M at k = 50 12.5 -> 3.7 ms, 1 M uniform points at k = 50 2.6 ->
// 0.65 ms, 1 M at k = 100 7.1 -> 2.1 ms, 100 k at k = 20 1.8 -> 0.2 ms (there
// single sparse queries held a lane for thousands of steps).
#include <type_traits>

#include "pgeof_device.hpp"
#include "pgeof_grid.hpp"
#include "pgeof_internal.hpp"

namespace pgeof_amd
{

namespace
{

// ------------------------------------------------- cross-lane helpers ----
// Keys are 64-bit: squared-distance bits << 32 | original index.  With the
// distance bits capped at the quiet NaN (0x7FC00000, above +inf) every key is
// the bit pattern of a finite non-negative double, and doubles order like
// their bits: keys compare with one v_cmp_lt_f64.
constexpr uint32_t kNanBits = 0x7FC00000u;
constexpr uint64_t kNoKey = 0x7FF0000000000000ull;  // +inf as a double: above every key

template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ uint64_t dpp(uint64_t v)
{
    return ((uint64_t)dpp<CTRL>((uint32_t)(v >> 32)) << 32) | dpp<CTRL>((uint32_t)v);
}
constexpr int quad_perm(int a, int b, int c, int d) { return a | (b << 2) | (c << 4) | (d << 6); }
constexpr int kRowShr = 0x110, kRowRor = 0x120, kRowMirror = 0x140, kRowHalfMirror = 0x141, kRowBcast15 = 0x142,
              kRowBcast31 = 0x143;

__device__ __forceinline__ uint32_t readlane(uint32_t v, uint32_t l)
{
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l);
}
__device__ __forceinline__ float readlane(float v, uint32_t l) { return __uint_as_float(readlane(__float_as_uint(v), l)); }
__device__ __forceinline__ int readlane(int v, uint32_t l) { return __builtin_amdgcn_readlane(v, (int)l); }
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ uint32_t from_lane(uint32_t v, uint32_t l)  // any lane's value, per lane
{
    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(l << 2), (int)v);
}
// set bits of m below this lane
__device__ __forceinline__ uint32_t lanes_below(uint64_t m)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// inclusive sum within rows of 16 lanes
__device__ __forceinline__ uint32_t row_scan(uint32_t v)
{
    v += dpp<kRowShr | 1>(v);
    v += dpp<kRowShr | 2>(v);
    v += dpp<kRowShr | 4>(v);
    v += dpp<kRowShr | 8>(v);
    return v;
}
// inclusive sum over the wave
__device__ __forceinline__ uint32_t wave_scan(uint32_t v)
{
    v = row_scan(v);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kRowBcast15, 0xA, 0xF, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kRowBcast31, 0xC, 0xF, false);
    return v;
}

// ------------------------------------------------------------- sorting ----
constexpr int kPerLane = 16;  // keys of a row that one lane sorts

// Batcher's odd-even merge sort of kPerLane keys: the comparators, in order
struct SortNet
{
    int n = 0;
    int a[64] = {}, b[64] = {};
    constexpr SortNet()
    {
        for (int p = 1; p < kPerLane; p *= 2)
            for (int q = p; q >= 1; q /= 2)
                for (int j = q % p; j + q < kPerLane; j += 2 * q)
                    for (int i = 0; i < q && i + j + q < kPerLane; ++i)
                        if ((i + j) / (2 * p) == (i + j + q) / (2 * p))
                        {
                            a[n] = i + j;
                            b[n] = i + j + q;
                            ++n;
                        }
    }
};
constexpr SortNet kNet16;
static_assert(kNet16.n == 63, "odd-even merge sort of 16");

// a, b = min, max.  (fmin and fmax would first quiet signalling NaNs, two
// more instructions; the keys are no NaNs.)
__device__ __forceinline__ void order2(double& a, double& b)
{
    double lo, hi;
    asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
    asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
    a = lo;
    b = hi;
}

template <int CTRL>
__device__ __forceinline__ double dpp(double v)
{
    return __longlong_as_double((long long)dpp<CTRL>((uint64_t)__double_as_longlong(v)));
}

// Rows of G * kPerLane keys, row r in lanes r * G .. r * G + G - 1, sorted
// ascending over (lane, register): every lane sorts its own keys, then runs
// of 1, 2, .. G lanes are merged (bitonic, first step mirrored).  A comparator
// within a lane is two instructions for 64 / G rows at once, so the sort of a
// row of 32 costs 8 instructions of the wave, of 64 about 31; sorting a row
// across 64 lanes, one key each, cost 115.
template <int CTRL, bool MIRROR>
__device__ __forceinline__ void lane_step(double v[kPerLane], bool keep_min)
{
    // two registers at a time: all sixteen partners at once would not leave
    // the candidates of the region in registers
#pragma unroll
    for (int r = 0; r < kPerLane / 2; ++r)
    {
        const int q = kPerLane - 1 - r;
        const double tr = dpp<CTRL>(v[MIRROR ? q : r]), tq = dpp<CTRL>(v[MIRROR ? r : q]);
        v[r] = (tr < v[r]) == keep_min ? tr : v[r];
        v[q] = (tq < v[q]) == keep_min ? tq : v[q];
        __builtin_amdgcn_sched_barrier(0);
    }
}
__device__ __forceinline__ void clean_lane(double v[kPerLane])
{
#pragma unroll
    for (int s = kPerLane / 2; s >= 1; s /= 2)
#pragma unroll
        for (int r = 0; r < kPerLane; ++r)
            if (!(r & s)) order2(v[r], v[r | s]);
}
template <int G>
__device__ __forceinline__ void sort_rows(double v[kPerLane], uint32_t lane)
{
#pragma unroll
    for (int c = 0; c < kNet16.n; ++c) order2(v[kNet16.a[c]], v[kNet16.b[c]]);
    const bool b0 = (lane & 1u) == 0, b1 = (lane & 2u) == 0, b2 = (lane & 4u) == 0;
    if constexpr (G >= 2)
    {
        lane_step<quad_perm(1, 0, 3, 2), true>(v, b0);
        clean_lane(v);
    }
    if constexpr (G >= 4)
    {
        lane_step<quad_perm(3, 2, 1, 0), true>(v, b1);
        lane_step<quad_perm(1, 0, 3, 2), false>(v, b0);
        clean_lane(v);
    }
    if constexpr (G >= 8)
    {
        lane_step<kRowHalfMirror, true>(v, b2);
        lane_step<quad_perm(2, 3, 0, 1), false>(v, b1);
        lane_step<quad_perm(1, 0, 3, 2), false>(v, b0);
        clean_lane(v);
    }
}

// ----------------------------------------------------------- selection ----
// NG * 64 candidates (distance bits b and index id in registers), of which
// the k nearest are wanted among at most `most` kept.  Absent ones have bits
// above every threshold tried (NaN or 0xFFFFFFFF).
template <int NG>
struct Candidates
{
    uint32_t b[NG], id[NG];

    __device__ __forceinline__ uint32_t count(uint32_t t) const
    {
        uint32_t c = 0;
#pragma unroll
        for (int u = 0; u < NG; ++u) c += (uint32_t)__popcll(__ballot(b[u] <= t));
        return c;
    }

    // A threshold tau with k <= n <= most candidates at or below it, first
    // tried at `guess`, by false position (counts grow about linearly with
    // the squared distance on a surface), then in turns by the next distance
    // above those that are too few, which settles ties, and by bisection of
    // the bits, which bounds the steps.
    // Thresholds up to `closed` are preferred (no point outside the scanned
    // cells is nearer); past it open = true, and `outer` bounds all distances
    // that are expected.  No threshold passes `limit` (a radius search's):
    // with fewer than k candidates up to it tau = limit and n < k.  Ties at
    // the k-th distance may leave no threshold: then n > most, tau is that
    // distance, and ties() bounds the indices.
    __device__ __forceinline__ uint32_t select(uint32_t k, uint32_t most, uint32_t guess, uint32_t closed,
                                               uint32_t outer, uint32_t limit, uint32_t& n, bool& open) const
    {
        const float target = 0.5f * (float)(k + most);
        int lo = -1, hi = 0;
        uint32_t clo = 0, chi = 0, cap = min(closed, limit);
        bool hi_known = false;
        open = false;
        uint32_t tau = min(guess, cap);
        for (int it = 0;; ++it)
        {
            const uint32_t c = count(tau);
            if (c < k)
            {
                lo = (int)tau, clo = c;
                if (tau == cap)
                {
                    if (cap == limit)
                    {
                        n = c;
                        return tau;
                    }
                    cap = cap < outer ? min(outer, limit) : limit;
                    open = true;
                }
            }
            else
            {
                hi = (int)tau, chi = c, hi_known = true;
                if (c <= most) break;
            }
            if (hi_known && hi - lo <= 1)
            {
                tau = (uint32_t)hi;
                break;
            }
            if (it >= 3 && (it & 1))
            {
                // no candidate lies between lo and the next one (if any)
                const uint32_t top = hi_known ? (uint32_t)hi : cap, up = next_above(lo);
                tau = up >= (uint32_t)(lo + 1) ? min(up, top) : top;
                lo = (int)tau - 1;
                continue;
            }
            float next;
            if (hi_known)
            {
                const float fl = lo < 0 ? 0.0f : __uint_as_float((uint32_t)lo), fh = __uint_as_float((uint32_t)hi);
                next = fl + (fh - fl) * ((target - (float)clo) * __builtin_amdgcn_rcpf((float)(chi - clo)));
            }
            else
                next = __uint_as_float(tau) *
                       fminf(fmaxf(target * __builtin_amdgcn_rcpf((float)max(c, 1u)), 1.2f), 16.0f);
            int nb = (int)uniform(__float_as_uint(next));
            const int top = hi_known ? hi - 1 : (int)cap;
            if (it >= 6) nb = hi_known ? lo + (hi - lo) / 2 : top;
            tau = (uint32_t)max(lo + 1, min(nb, top));
        }
        n = chi;
        // every candidate kept: the farthest one bounds the search
        return tau < 0x7F800000u ? tau : min(tau, largest());
    }

    // of one value per lane
    __device__ __forceinline__ static uint32_t wave_max(uint32_t m)
    {
        m = max(m, dpp<kRowShr | 1>(m));
        m = max(m, dpp<kRowShr | 2>(m));
        m = max(m, dpp<kRowShr | 4>(m));
        m = max(m, dpp<kRowShr | 8>(m));
        return max(max(readlane(m, 15u), readlane(m, 31u)), max(readlane(m, 47u), readlane(m, 63u)));
    }

    __device__ __forceinline__ uint32_t largest() const
    {
        uint32_t m = 0;
#pragma unroll
        for (int u = 0; u < NG; ++u) m = max(m, b[u] > kNanBits ? 0u : b[u]);
        return wave_max(m);
    }

    // the smallest distance bits above lo (>= -1); less than that if none are
    __device__ __forceinline__ uint32_t next_above(int lo) const
    {
        uint32_t m = 0xFFFFFFFFu;
#pragma unroll
        for (int u = 0; u < NG; ++u) m = min(m, b[u] - (uint32_t)(lo + 1));  // those below wrap around
        return ~wave_max(~m) + (uint32_t)(lo + 1);
    }

    // Of the candidates exactly at tau, those with index <= the result, with
    // the nearer ones, are at least k and at most `most`: n.  By bisection of
    // the indices from the highest bit of the largest one; any number in that
    // range ends it (after about 5 steps; exactly k took all 32).
    __device__ __forceinline__ uint32_t ties(uint32_t k, uint32_t most, uint32_t tau, uint32_t top_bit, uint32_t& n) const
    {
        const uint32_t nearer = tau ? count(tau - 1u) : 0u;
        uint32_t tied[NG];
#pragma unroll
        for (int u = 0; u < NG; ++u) tied[u] = b[u] == tau ? id[u] : 0xFFFFFFFFu;
        uint32_t t = 0;
        for (uint32_t bit = top_bit;; bit >>= 1)
        {
            // t: fewer than k with the tied indices below it
            uint32_t c = nearer;
#pragma unroll
            for (int u = 0; u < NG; ++u) c += (uint32_t)__popcll(__ballot(tied[u] < (t | bit)));
            if (c < k)
                t |= bit;
            else if (c <= most)
            {
                n = c;
                return (t | bit) - 1u;
            }
            if (bit <= 1u) break;
        }
        n = k;
        return t;
    }

    // the kept candidates as keys to LDS
    template <class In>
    __device__ __forceinline__ void store_if(uint64_t* dst, In in) const
    {
        uint32_t n = 0;
#pragma unroll
        for (int u = 0; u < NG; ++u)
        {
            const bool keep = in(b[u], id[u]);
            const uint64_t m = __ballot(keep);
            if (keep) dst[n + lanes_below(m)] = ((uint64_t)b[u] << 32) | id[u];
            n += (uint32_t)__popcll(m);
        }
    }
    // ... of a threshold and its n; returns the number kept, and in `last` the
    // largest index kept of those at the threshold
    __device__ __forceinline__ uint32_t store(uint64_t* dst, uint32_t k, uint32_t most, uint32_t tau, uint32_t n,
                                              uint32_t top_bit, uint32_t& last) const
    {
        last = 0xFFFFFFFFu;
        if (n <= most)
        {
            store_if(dst, [&](uint32_t bb, uint32_t) { return bb <= tau; });
            return n;
        }
        const uint32_t tie = ties(k, most, tau, top_bit, n);
        store_if(dst, [&](uint32_t bb, uint32_t i) { return bb < tau || (bb == tau && i <= tie); });
        last = tie;
        return n;
    }
};

// --------------------------------------------------------- the kernel ----
// A level of the table, read with scalar loads (the table was written by
// earlier kernels and does not change during this one).
#define PGEOF_CONST __attribute__((address_space(4)))
__device__ __forceinline__ const PGEOF_CONST Level* scalar_level(const LevelTable* tab, uint32_t l)
{
    return (const PGEOF_CONST Level*)(tab->lv + l);
}

// Candidates of a cell's 3x3x3 cube kept in registers, in groups of 64 (one
// per lane); larger cubes are streamed instead.
template <int G>
constexpr uint32_t kGroupsOf = G <= 2 ? 6 : 12;
// Streamed candidates collected in LDS before the farthest are dropped.
constexpr uint32_t kBufGroups = 6, kBufKeys = 64 * kBufGroups;
constexpr uint32_t kAhead = 3;  // groups of 64 of them loaded together

// Block b's place in the sorted order of the queries.  Runs of kRun blocks go
// to the XCDs in turn: a run's queries are neighbours and share their XCD's
// L2, and the sparse parts of a scene, which cost more per query, spread over
// all XCDs (one contiguous eighth per XCD: 10 M LiDAR points at k = 20 took
// 15.6 ms instead of 12.3, the XCDs of the dense parts idle at the end).  The
// runs are taken from both ends of the order inwards: the lowest and highest
// points of a scene are its sparsest, and what runs longest starts first (the
// lowest ones taken last ran on for 3 ms after all others).
__device__ __forceinline__ uint32_t work_block(uint32_t b, uint32_t nb)
{
    constexpr uint32_t kXcd = 8, kRun = 32;
    const uint32_t whole = nb / (kXcd * kRun) * (kXcd * kRun);
    uint32_t l = b;
    if (b < whole)
    {
        const uint32_t x = b % kXcd, s = b / kXcd;
        l = (s / kRun * kXcd + x) * kRun + s % kRun;
    }
    // of eight runs in a row four come from either end, and an XCD's runs
    // from both ends in turn
    const uint32_t runs = nb / kRun, j = l / kRun, e = l % kRun;
    if (j >= runs) return nb / (2 * kRun) * kRun + (runs & 1u) * kRun + e;
    uint32_t side = j & 1u, at = j / 2;
    if (j < runs / kXcd * kXcd)
    {
        const uint32_t x = j % kXcd, g = j / kXcd;
        side = (x + g) & 1u;
        at = g * (kXcd / 2) + x / 2;
    }
    return side ? nb - kRun - at * kRun + e : at * kRun + e;
}

// G: lanes that sort one query's row of kPerLane * G kept candidates.
// WAVES per SIMD: with three (168 registers) nothing spills but scalars (up to
// three vector registers of the radius modes).  With four (128 registers) four
// or five spill, which k = 9 to 27 repay where the launch keeps four waves on
// every SIMD (us per call, fused, three / four: 10 M LiDAR points at k = 20, mean
// of eight clouds, 7650 / 7310; 1 M 946 / 917; 1 M uniform points 717 / 685; 300 k
// 291 / 280; 10 k 75.8 / 79.4); k <= 8 is slower with four (1 M LiDAR points at k =
// 8 762 / 784), larger rows do not fit.
template <int MODE, int G, int WAVES>
__global__ __launch_bounds__(64, WAVES) void k_wave_search(WaveArgs a)
{
    constexpr bool RADIUS = MODE == kModeRadius || MODE == kModeRadiusCsr;
    if (!RADIUS && a.other && *a.other) return;
    constexpr uint32_t kGroups = kGroupsOf<G>;
    constexpr uint32_t kMost = (uint32_t)(kPerLane * G);  // candidates kept per query
    constexpr uint32_t kBatch = 64 / G;                   // queries collected before their rows are sorted
    constexpr uint32_t kStride = kMost + 1;               // odd: the rows start on different LDS banks
    __shared__ uint64_t lds[kBatch * kStride + kBufKeys];
    uint64_t* const kept = lds;
    uint64_t* const buf = lds + kBatch * kStride;
    const uint32_t lane = threadIdx.x;
    const uint32_t k = a.k;

    // Queries t0 .. t0 + nq.  Radius searches: the 64 / q_per_wave waves of
    // a group look at its 64 queries first; if those are sparse, the first
    // wave takes them all.
    const uint32_t wave = work_block(blockIdx.x, gridDim.x), members = RADIUS ? 64u / a.q_per_wave : 1u;
    uint32_t t0 = RADIUS ? wave / members * 64u : wave * a.q_per_wave;
    uint32_t nq = min(RADIUS ? 64u : a.q_per_wave, a.n_query - t0);
    const uint32_t nl = uniform((uint32_t)a.tab->n_levels);

    // lane group l (16 lanes) looks after pyramid level l
    const Level* __restrict__ LV = &a.tab->lv[min(lane >> 4, nl - 1)];
    const float inv_h = (float)LV->inv_h;
    const int g0 = LV->g[0], g1 = LV->g[1], g2 = LV->g[2];
    const uint32_t* __restrict__ cs = LV->cs;
    // rows of a region: lanes 0..8 of each group
    const uint32_t rr = lane & 15u;
    const int row_dy = (int)(rr % 3u) - 1, row_dz = (int)(rr / 3u) - 1;
    const bool row_ok = (lane >> 4) < nl && rr < 9u;

    // This lane's query.  Its region is found in float, relative to the
    // grid's origin: a cell off by one at a cell's face, or the slack of the
    // region's faces, changes no result.
    const uint32_t limit = RADIUS ? a.limit : kNanBits;
    float4 qv;
    uint64_t finite;
    float relx, rely, relz, slack;
    auto load_queries = [&]() {
        qv = make_float4(0.f, 0.f, 0.f, 0.f);
        if (lane < nq) qv = a.queries[t0 + lane];
        finite = __ballot(isfinite(qv.x) && isfinite(qv.y) && isfinite(qv.z));
        if (RADIUS && limit == 0xFFFFFFFFu) finite = 0;  // no distance is below the radius
        const PGEOF_CONST Level* L0 = scalar_level(a.tab, 0);
        relx = (float)((double)qv.x - L0->lo[0]), rely = (float)((double)qv.y - L0->lo[1]),
        relz = (float)((double)qv.z - L0->lo[2]);
        // rounding of a difference of such a coordinate and a cell's face
        slack = 5e-7f * (fmaxf(fabsf(relx), fmaxf(fabsf(rely), fabsf(relz))) +
                         (float)(L0->h * (double)max(L0->g[0], max(L0->g[1], L0->g[2]))));
    };
    load_queries();
    auto cell32 = [](float rel, float ih, int g) -> int {
        return (int)fminf(fmaxf(rel * ih, 0.0f), (float)(g - 1));
    };

    // How far the 3x3x3 cells around cell (c0, c1, c2) of a level cover this
    // lane's query: distance bits up to which a ball around it stays inside
    // them (faces on the grid's border do not count), and bits no distance to
    // a point in them exceeds.
    auto cover = [&](int c0, int c1, int c2, float h, int a0, int a1, int a2, uint32_t& inner, uint32_t& all) {
        const float xl = relx - (float)(c0 - 1) * h, xh = (float)(c0 + 2) * h - relx;
        const float yl = rely - (float)(c1 - 1) * h, yh = (float)(c1 + 2) * h - rely;
        const float zl = relz - (float)(c2 - 1) * h, zh = (float)(c2 + 2) * h - relz;
        float g = INFINITY;
        g = c0 > 1 ? fminf(g, xl) : g;
        g = c0 < a0 - 2 ? fminf(g, xh) : g;
        g = c1 > 1 ? fminf(g, yl) : g;
        g = c1 < a1 - 2 ? fminf(g, yh) : g;
        g = c2 > 1 ? fminf(g, zl) : g;
        g = c2 < a2 - 2 ? fminf(g, zh) : g;
        const float gm = fmaxf(g - h * a.margin - slack, 0.0f);
        inner = g == INFINITY ? kNanBits : __float_as_uint(gm * gm * 0.99996f);
        const float ex = fmaxf(xl, xh), ey = fmaxf(yl, yh), ez = fmaxf(zl, zh);
        all = __float_as_uint((ex * ex + ey * ey + ez * ez) * 1.001f);
    };

    // Sorted rows of the queries first .. first + count, `stride` keys apart
    // in LDS; lane s holds the number of keys of query first + s.
    auto write_rows = [&](uint32_t first, uint32_t count, uint32_t stride, uint32_t keys) {
        auto store_key = [&](uint32_t* oi, float* od, uint32_t e, uint64_t key, uint32_t hits) {
            const bool none = RADIUS ? e >= hits : key == kNoKey;
            oi[e] = none ? 0xFFFFFFFFu : (uint32_t)key;
            // past the hits 0, and r^2 in the last slot (nanoflann's
            // RKNNResultSet::init)
            const float pad = !RADIUS ? INFINITY : (e == k - 1 ? a.r2 : 0.0f);
            if (od) od[e] = none ? pad : __uint_as_float((uint32_t)(key >> 32));
        };
        if (RADIUS && k <= 32)
        {
            // two rows per store, one per half of the wave
            const uint32_t e = lane & 31u;
#pragma unroll 4
            for (uint32_t s = lane >> 5; s < ((count + 1) & ~1u); s += 2)
            {
                const uint32_t qorig = from_lane(__float_as_uint(qv.w), (first + s) & 63u);
                const uint32_t hits = min(from_lane(keys, s & 63u), k);
                if (s < count && e < (MODE == kModeRadiusCsr ? hits : k))
                    store_key(a.out_idx + (size_t)qorig * k, a.out_d2 ? a.out_d2 + (size_t)qorig * k : nullptr, e,
                              lds[s * stride + min(e, stride - 1u)], hits);
            }
        }
        else
        {
#pragma unroll 4
            for (uint32_t s = 0; s < count; ++s)
            {
                const uint32_t qorig = readlane(__float_as_uint(qv.w), first + s);
                uint32_t* oi = a.out_idx + (size_t)qorig * k;
                float* od = a.out_d2 ? a.out_d2 + (size_t)qorig * k : nullptr;
                const uint32_t hits = RADIUS ? min(readlane(keys, s), k) : k;
#pragma unroll
                for (uint32_t e0 = 0; e0 < kMost; e0 += 64)
                {
                    const uint32_t e = e0 + lane;
                    if (e >= (MODE == kModeRadiusCsr ? hits : k)) continue;
                    store_key(oi, od, e, lds[s * stride + min(e, stride - 1u)], hits);
                }
            }
        }
        if (RADIUS && a.out_count)
        {
            // lane s counts the hits of query first + s
            const uint32_t qorig = from_lane(__float_as_uint(qv.w), (first + lane) & 63u);
            if (lane < count) a.out_count[qorig] = min(keys, k);
        }
    };

    if constexpr (RADIUS)
    {
        // Queries with few points around them and at most 16 hits each: one
        // per lane, its region's points one after the other (1 M
        // uniform points with their own point in the ball: a wave per query
        // would spend its instructions on one candidate).
        const PGEOF_CONST Level* L = scalar_level(a.tab, nl - 1);
        const float h = (float)L->h, ih = (float)L->inv_h;
        const int a0 = L->g[0], a1 = L->g[1], a2 = L->g[2];
        const uint32_t* __restrict__ tcs = L->cs;
        const float4* __restrict__ pts = L->pts;
        const int cx = cell32(relx, ih, a0), cy = cell32(rely, ih, a1), cz = cell32(relz, ih, a2);
        const bool mine = (finite >> lane) & 1ull;
        // The part of the 27 cells that the ball can meet: where the cap of the
        // grid makes its cells larger than the radius, about two of the nine
        // rows (1 M uniform points, r = 0.2, cap 30: 352 us per call with all
        // nine, 279 now; 1 M LiDAR points, r = 0.02, cap 24: 438, 307).
        const float reach = sqrtf(__uint_as_float(min(limit, 0x7F800000u))) * 1.00001f;
        int x0 = max(cx - 1, 0), x1 = min(cx + 1, a0 - 1), y0 = max(cy - 1, 0), y1 = min(cy + 1, a1 - 1),
            z0 = max(cz - 1, 0), z1 = min(cz + 1, a2 - 1);
        if (h > 1.25f * reach)
        {
            const float w = reach + slack + h * a.margin;
            x0 = max(x0, cell32(relx - w, ih, a0)), x1 = min(x1, cell32(relx + w, ih, a0));
            y0 = max(y0, cell32(rely - w, ih, a1)), y1 = min(y1, cell32(rely + w, ih, a1));
            z0 = max(z0, cell32(relz - w, ih, a2)), z1 = min(z1, cell32(relz + w, ih, a2));
        }
        const int ny = y1 - y0 + 1, n_rows = mine ? ny * (z1 - z0 + 1) : 0;
        // the first cell of the rows one after the other, ny per layer
        struct Rows
        {
            uint32_t at, step, skip;
            int y, ny;
            __device__ __forceinline__ void next()
            {
                at += step;
                if (++y == ny) y = 0, at += skip;
            }
        };
        auto rows_from = [&](uint32_t first, int n) {
            return Rows{first, (uint32_t)a0, (uint32_t)(a1 - n) * (uint32_t)a0, 0, n};
        };
        const uint32_t first_row = ((uint32_t)z0 * (uint32_t)a1 + (uint32_t)y0) * (uint32_t)a0;
        uint32_t around = 0, rows = 0;  // points in them, rows that hold some
        Rows R = rows_from(first_row, ny);
#pragma unroll
        for (int r = 0; r < 9; ++r, R.next())
        {
            if (__ballot(r < n_rows) == 0) break;
            if (r < n_rows)
            {
                const uint32_t c = gload(tcs, R.at + (uint32_t)x1 + 1u) - gload(tcs, R.at + (uint32_t)x0);
                around += c;
                rows += c ? 1u : 0u;
            }
        }
        uint32_t inner, all;
        cover(cx, cy, cz, h, a0, a1, a2, inner, all);
        // No more than 16 around any: no more hits, the first wave's work.
        // Else each wave of the group looks at its own queries, q0 .. q0 + n_own
        // (all 64 scanned by each, the first to write them: 2 M uniform points
        // with 8 hits, cap 24, 895 us, now 847).
        const bool alone = members == 1 || __ballot(mine && (around > (uint32_t)kPerLane || inner < limit)) == 0;
        if (alone && wave % members) return;
        const uint32_t q0 = alone ? 0u : wave % members * a.q_per_wave;
        if (q0 >= nq) return;
        const uint32_t n_own = alone ? nq : min(a.q_per_wave, nq - q0);
        const bool own = mine && lane - q0 < n_own;
        constexpr uint32_t kFew = 80;  // points a lane looks at
        uint32_t n = 0;
        constexpr uint32_t kSparse = (uint32_t)kPerLane + 1;
        static_assert(64 * kSparse <= sizeof(lds) / 8, "rows of the sparse case");
        uint64_t* row = lds + ((lane - q0) & 63u) * kSparse;
        const int own_rows = own ? n_rows : 0;
        if (__ballot(own && (around > kFew || inner < limit)) == 0)
        {
            Rows S = rows_from(first_row, ny);
#pragma unroll 1
            for (int r = 0; r < 9; ++r, S.next())
            {
                if (__ballot(r < own_rows) == 0) break;
                uint32_t j = 0, e = 0;
                if (r < own_rows)
                {
                    j = gload(tcs, S.at + (uint32_t)x0);
                    e = gload(tcs, S.at + (uint32_t)x1 + 1u);
                }
                for (; j < e; j += 4)
                {
                    float4 p[4];
#pragma unroll
                    for (uint32_t u = 0; u < 4; ++u) p[u] = gload(pts, min(j + u, e - 1u));
#pragma unroll
                    for (uint32_t u = 0; u < 4; ++u)
                    {
                        const uint32_t d = min(__float_as_uint(sqdist32(qv.x, qv.y, qv.z, p[u].x, p[u].y, p[u].z)), kNanBits);
                        if (j + u < e && d <= limit)
                        {
                            if (n < (uint32_t)kPerLane) row[n] = ((uint64_t)d << 32) | __float_as_uint(p[u].w);
                            ++n;
                        }
                    }
                }
            }
        }
        else
            n = (uint32_t)kPerLane + 1u;
        if (__ballot(own && n > (uint32_t)kPerLane) == 0)
        {
            double v[kPerLane];
#pragma unroll
            for (int r = 0; r < kPerLane; ++r) v[r] = __longlong_as_double((long long)((uint32_t)r < n ? row[r] : kNoKey));
            sort_rows<1>(v, lane);
#pragma unroll
            for (int r = 0; r < kPerLane; ++r) row[r] = (uint64_t)__double_as_longlong(v[r]);
            wave_sync();
            write_rows(q0, n_own, kSparse, from_lane(n, (lane + q0) & 63u));
            return;
        }
        // Up to 32 hits each: two lanes per query, 32 queries at a time, one
        // lane filling a row from the front, the other from its end (200 k
        // uniform points, 20 hits, cap 30: 241 us per call with a wave per query,
        // 190 so; cap 64: 269, 203).
        if (members <= 2)
        {
            // Points per row of cells up to which 32 hits are likely enough
            // to try: 32 in the ball are 23 per row in a volume, 31 on a
            // horizontal plane; in a volume one of 32 queries is past them
            // from 22 hits on average, 16 per row.  (224 per region whatever
            // its rows: 1 M LiDAR points with 50 hits spent 64 us more on tries
            // that failed; 24 per row in a volume too: 2 M uniform points with
            // 28 hits 1813 us, now 1550.)
            constexpr uint32_t kFewPair = 24, kFewVolume = 18;
            constexpr uint32_t kPair = 2 * kPerLane, kPairStride = kPair + 1;
            static_assert(32 * kPairStride <= sizeof(lds) / 8, "rows of the pairs");
            const uint32_t odd = lane & 1u;
            uint64_t* prow = lds + (lane >> 1) * kPairStride;
            bool done = true;
#pragma unroll 1
            for (uint32_t first = q0; first < q0 + n_own; first += 32)
            {
                const uint32_t count = min(32u, q0 + n_own - first), ql = (first + (lane >> 1)) & 63u;
                done = __ballot(own && lane - first < count &&
                                (around > (rows > 5 ? kFewVolume : kFewPair) * rows || inner < limit)) == 0;
                if (!done) break;
                const float x = __uint_as_float(from_lane(__float_as_uint(qv.x), ql)),
                            y = __uint_as_float(from_lane(__float_as_uint(qv.y), ql)),
                            z = __uint_as_float(from_lane(__float_as_uint(qv.z), ql));
                const int px0 = (int)from_lane((uint32_t)x0, ql), px1 = (int)from_lane((uint32_t)x1, ql),
                          p_rows = (int)from_lane(lane - first < count ? (uint32_t)n_rows : 0u, ql);
                Rows S = rows_from(from_lane(first_row, ql), (int)from_lane((uint32_t)ny, ql));
                uint32_t got = 0;
#pragma unroll 1
                for (int r = 0; r < 9; ++r, S.next())
                {
                    if (__ballot(r < p_rows) == 0) break;
                    uint32_t j = 0, e = 0;
                    if (r < p_rows)
                    {
                        j = gload(tcs, S.at + (uint32_t)px0) + 4u * odd;
                        e = gload(tcs, S.at + (uint32_t)px1 + 1u);
                    }
                    for (; j < e; j += 8)
                    {
                        float4 p[4];
#pragma unroll
                        for (uint32_t u = 0; u < 4; ++u) p[u] = gload(pts, min(j + u, e - 1u));
#pragma unroll
                        for (uint32_t u = 0; u < 4; ++u)
                        {
                            const uint32_t d = min(__float_as_uint(sqdist32(x, y, z, p[u].x, p[u].y, p[u].z)), kNanBits);
                            if (j + u < e && d <= limit)
                            {
                                if (got < kPair)
                                    prow[odd ? kPair - 1 - got : got] = ((uint64_t)d << 32) | __float_as_uint(p[u].w);
                                ++got;
                            }
                        }
                    }
                }
                const uint32_t other = from_lane(got, lane ^ 1u), both = got + other;
                done = __ballot(both > kPair) == 0;
                if (!done) break;
                wave_sync();
                const uint32_t front = odd ? other : got, back = both - front;
                double v[kPerLane];
#pragma unroll
                for (int r = 0; r < kPerLane; ++r)
                {
                    const uint32_t i = odd * kPerLane + (uint32_t)r;
                    v[r] = __longlong_as_double((long long)(i < front || i >= kPair - back ? prow[i] : kNoKey));
                }
                sort_rows<2>(v, lane);
#pragma unroll
                for (int r = 0; r < kPerLane; ++r) prow[odd * kPerLane + r] = (uint64_t)__double_as_longlong(v[r]);
                wave_sync();
                write_rows(first, count, kPairStride, from_lane(both, (2 * lane) & 63u));
                wave_sync();
            }
            if (done) return;
        }
        if (members > 1)
        {
            t0 += wave % members * a.q_per_wave;
            if (t0 >= a.n_query) return;
            nq = min(a.q_per_wave, a.n_query - t0);
            load_queries();
        }
    }

    // the current region: the 3x3x3 cells around one of level rl
    uint64_t served = 0;  // queries in that cell
    uint32_t rl = 0;
    int rx = 0, ry = 0, rz = 0;  // the cell
    uint32_t total = 0;          // candidates in the region
    bool in_regs = false;
    uint32_t closed = 0, outer = 0;  // how far it covers this lane's query
    float px[kGroups], py[kGroups], pz[kGroups];
    uint32_t pi[kGroups];
#pragma unroll
    for (uint32_t u = 0; u < kGroups; ++u) px[u] = py[u] = pz[u] = 0.f, pi[u] = 0;
    uint32_t guess = 0;  // distance bits expected to keep about `target` candidates
    const float target = 0.5f * (float)(k + kMost);

    // The next region's rows of cells on every level, looked up while the
    // queries of the current one are searched: cell, points of this lane's row
    int ncx = 0, ncy = 0, ncz = 0;
    uint32_t n_st = 0, n_end = 0;
    auto look_up = [&](uint32_t i) {
        ncx = cell32(readlane(relx, i), inv_h, g0), ncy = cell32(readlane(rely, i), inv_h, g1),
        ncz = cell32(readlane(relz, i), inv_h, g2);
        const int y = ncy + row_dy, z = ncz + row_dz;
        n_st = n_end = 0;
        if (row_ok && (uint32_t)y < (uint32_t)g1 && (uint32_t)z < (uint32_t)g2)
        {
            const uint32_t at = ((uint32_t)z * (uint32_t)g1 + (uint32_t)y) * (uint32_t)g0;
            n_st = gload(cs, at + (uint32_t)max(ncx - 1, 0));
            n_end = gload(cs, at + (uint32_t)min(ncx + 1, g0 - 1) + 1u);
        }
    };
    if (finite) look_up((uint32_t)__ffsll((unsigned long long)finite) - 1u);

    for (uint32_t base = 0; base < nq; base += kBatch)
    {
        const uint32_t nb = min(kBatch, nq - base);
        uint32_t n_kept = 0;  // of query base + lane
        for (uint32_t s = 0; s < nb; ++s)
        {
            const uint32_t i = base + s;
            if (!((finite >> i) & 1ull)) continue;  // keeps nothing
            const float qxf = readlane(qv.x, i), qyf = readlane(qv.y, i), qzf = readlane(qv.z, i);
            uint64_t* row = kept + s * kStride;
            if (!((served >> i) & 1ull))
            {
                // ---- a new region: every level's rows are at hand ----
                const int cx = ncx, cy = ncy, cz = ncz;
                const uint32_t st = n_st, len = n_end - n_st;
                const uint32_t incl = row_scan(len);
                // the finest level whose region holds a.need points; a finer
                // one with k points if that region does not fit the registers
                uint32_t prev = 0;
                for (rl = 0;; ++rl)
                {
                    total = readlane(incl, 16u * rl + 15u);
                    if (total >= a.need || rl + 1 >= nl) break;
                    prev = total;
                }
                if (total > 64u * kGroups && prev >= k) --rl, total = prev;
                const uint32_t gl = 16u * rl;
                rx = readlane(cx, gl), ry = readlane(cy, gl), rz = readlane(cz, gl);
                in_regs = (RADIUS || total >= k) && total <= 64u * kGroups;
                const PGEOF_CONST Level* L = scalar_level(a.tab, rl);
                if (in_regs)
                {
                    const float4* __restrict__ pts = L->pts;
                    const uint32_t first = incl - len, off = st - first;
                    uint32_t start[9];
#pragma unroll
                    for (uint32_t r = 1; r < 9; ++r) start[r] = readlane(first, gl + r);
#pragma unroll
                    for (uint32_t u = 0; u < kGroups; ++u)
                        if (u * 64u < total)
                        {
                            // row of candidate f: the last one that starts at
                            // or before it; past the last candidate NaN
                            const uint32_t f = min(u * 64u + lane, total - 1u);
                            uint32_t r = gl;
#pragma unroll
                            for (uint32_t v = 1; v < 9; ++v) r += f >= start[v] ? 1u : 0u;
                            const float4 p = gload(pts, f + from_lane(off, r));
                            px[u] = u * 64u + lane < total ? p.x : __uint_as_float(kNanBits);
                            py[u] = p.y, pz[u] = p.z, pi[u] = __float_as_uint(p.w);
                        }
                        else
                            px[u] = __uint_as_float(kNanBits);
                }
                const float h = (float)L->h, ih = (float)L->inv_h;
                const int a0 = L->g[0], a1 = L->g[1], a2 = L->g[2];
                served = __ballot(cell32(relx, ih, a0) == rx && cell32(rely, ih, a1) == ry &&
                                  cell32(relz, ih, a2) == rz) |
                         (1ull << i);
                cover(rx, ry, rz, h, a0, a1, a2, closed, outer);
                const uint64_t later = finite & ~served & (~0ull << i);
                if (later) look_up((uint32_t)__ffsll((unsigned long long)later) - 1u);
            }

            uint32_t n = 0;           // candidates kept
            uint32_t tau = kNanBits;  // threshold they were kept by
            bool done = false, bounded = false;
            if (in_regs)
            {
                // ---- candidates in registers ----
                if (guess == 0)
                {
                    // an even spread over the region's area
                    const float h = (float)scalar_level(a.tab, rl)->h;
                    guess = uniform(__float_as_uint(h * h * 2.8f * target / (float)max(total, 1u)));
                }
                auto search = [&](auto groups) {
                    constexpr int NG = decltype(groups)::value;
                    Candidates<NG> c;
#pragma unroll
                    for (int u = 0; u < NG; ++u)
                    {
                        c.b[u] = __float_as_uint(sqdist32(qxf, qyf, qzf, px[u], py[u], pz[u]));
                        c.id[u] = pi[u];
                    }
                    bool open;
                    tau = c.select(k, kMost, guess, readlane(closed, i), readlane(outer, i), limit, n, open);
                    bounded = tau < 0x7F800000u;
                    done = bounded && !open;
                    uint32_t tie;
                    if (done) n = c.store(row, k, kMost, tau, n, a.top_bit, tie);
                };
                if (total <= 64u)
                    search(std::integral_constant<int, 1>{});
                else if (total <= 128u)
                    search(std::integral_constant<int, 2>{});
                else if (total <= 192u)
                    search(std::integral_constant<int, 3>{});
                else if (total <= 256u)
                    search(std::integral_constant<int, 4>{});
                else if (kGroups == 6 || total <= 384u)
                    search(std::integral_constant<int, 6>{});
                else if (total <= 512u)
                    search(std::integral_constant<int, (kGroups > 6 ? 8 : 6)>{});
                else
                    search(std::integral_constant<int, (int)kGroups>{});
            }
            if (!done)
            {
                // ---- the cells of the level that meet the ball of tau.  With
                // no threshold at hand (fewer than k candidates, or too many
                // for the registers) it is taken from the last query's, or an
                // even spread over the region, and grows until the ball holds
                // k points: then it holds the k nearest ones. ----
                const PGEOF_CONST Level* L = scalar_level(a.tab, rl);
                const double lo0 = L->lo[0], lo1 = L->lo[1], lo2 = L->lo[2], h = L->h, ih = L->inv_h;
                const int a0 = L->g[0], a1 = L->g[1], a2 = L->g[2];
                const uint32_t* __restrict__ ucs = L->cs;
                const float4* __restrict__ pts = L->pts;
                const double margin = h * (double)a.margin;
                const double qx = qxf, qy = qyf, qz = qzf;
                double away = 0.0;  // of the query from the grid's box
                if (!bounded)
                {
                    const double dx = fmax(fmax(lo0 - qx, qx - (lo0 + (double)a0 * h)), 0.0),
                                 dy = fmax(fmax(lo1 - qy, qy - (lo1 + (double)a1 * h)), 0.0),
                                 dz = fmax(fmax(lo2 - qz, qz - (lo2 + (double)a2 * h)), 0.0);
                    away = sqrt(dx * dx + dy * dy + dz * dz);
                    const double w = guess > 0 && guess < 0x7F800000u
                                         ? 1.25 * (double)__uint_as_float(guess)
                                         : h * h * 2.8 * (double)target / (double)max(total, 1u);
                    const double r = fmax(sqrt(w), away + 0.25 * h);
                    const uint32_t t = uniform(__float_as_uint((float)(r * r)));
                    tau = min(t < 0x7F800000u ? t : kNanBits, limit);
                }
                Box B{0, 0, 0, 0, 0, 0};
                uint32_t ny = 1, nr = 1;
                double lim = INFINITY;  // squared distance of the rows of interest
                // rows from the query's own outwards
                const int yc = cell_coord(qy, lo1, ih, a1), zc = cell_coord(qz, lo2, ih, a2);
                auto row_gap2 = [&](uint32_t r, int& y, int& z) -> double {
                    z = nth_near((int)(r / ny), zc, B.z0, B.z1), y = nth_near((int)(r % ny), yc, B.y0, B.y1);
                    const double dz = axis_gap(qz, z, lo2, h, margin), dy = axis_gap(qy, y, lo1, h, margin);
                    return dz * dz + dy * dy;
                };
                auto row_range = [&](int y, int z, int xa, int xb, uint32_t& st, uint32_t& len) {
                    const uint32_t at = ((uint32_t)z * (uint32_t)a1 + (uint32_t)y) * (uint32_t)a0;
                    st = gload(ucs, at + (uint32_t)xa);
                    len = gload(ucs, at + (uint32_t)xb + 1u) - st;
                };
                // of the points exactly at tau those with an index up to `tie`
                // are collected
                uint32_t tie = 0xFFFFFFFFu;
                for (;;)
                {
                    const float w = __uint_as_float(tau);
                    lim = w < INFINITY ? (double)w * 1.00001 + 1e-37 : INFINITY;
                    const double ext = sqrt(lim) + margin;
                    B = Box{cell_coord(qx - ext, lo0, ih, a0), cell_coord(qx + ext, lo0, ih, a0),
                            cell_coord(qy - ext, lo1, ih, a1), cell_coord(qy + ext, lo1, ih, a1),
                            cell_coord(qz - ext, lo2, ih, a2), cell_coord(qz + ext, lo2, ih, a2)};
                    B.y0 = (int)uniform((uint32_t)B.y0), B.y1 = (int)uniform((uint32_t)B.y1);
                    B.z0 = (int)uniform((uint32_t)B.z0), B.z1 = (int)uniform((uint32_t)B.z1);
                    ny = (uint32_t)(B.y1 - B.y0 + 1), nr = ny * (uint32_t)(B.z1 - B.z0 + 1);
                    uint32_t n_buf = 0;
                    bool again = false;
                    // the nearest of the collected keys stay (at least k, at
                    // most kMost of them), tau and tie drop to their bound.
                    // (With the distance alone every further point of a spot
                    // of coincident ones was collected again: 200 k LiDAR
                    // points, 20 k of them at the origin, k = 20, 25.9 ms per
                    // call; 2.5 now, the heaps of the general search 7.2.)
                    auto reduce = [&]() {
                        wave_sync();
                        Candidates<(int)kBufGroups> c;
#pragma unroll
                        for (uint32_t u = 0; u < kBufGroups; ++u)
                        {
                            const uint64_t key = u * 64u + lane < n_buf ? buf[u * 64u + lane] : ~0ull;
                            c.b[u] = (uint32_t)(key >> 32), c.id[u] = (uint32_t)key;
                        }
                        wave_sync();
                        bool open;
                        uint32_t m;
                        const float t = __uint_as_float(tau) * target * __builtin_amdgcn_rcpf((float)n_buf);
                        tau = c.select(k, kMost, uniform(__float_as_uint(t)), kNanBits, kNanBits, kNanBits, m, open);
                        n_buf = c.store(buf, k, kMost, tau, m, a.top_bit, tie);
                    };
                    // one row of cells per lane, then the rows' points as one
                    // list spread over the lanes, kAhead groups loaded together
                    for (uint32_t r0 = 0; r0 < nr && !again; r0 += 64)
                    {
                        uint32_t st = 0, len = 0;
                        const uint32_t r = r0 + lane;
                        if (r < nr)
                        {
                            int y, z;
                            const double rem = lim - row_gap2(r, y, z);
                            int xa = B.x0, xb = rem < 0.0 ? xa - 1 : B.x1;
                            if (rem >= 0.0 && rem < INFINITY)
                            {
                                const double xr = sqrt(rem) + margin;
                                xa = max(xa, cell_coord(qx - xr, lo0, ih, a0));
                                xb = min(xb, cell_coord(qx + xr, lo0, ih, a0));
                            }
                            if (xa <= xb) row_range(y, z, xa, xb, st, len);
                        }
                        const uint32_t incl = wave_scan(len), first = incl - len, off = st - first;
                        const uint32_t tot = readlane(incl, 63u);
                        for (uint32_t f0 = 0; f0 < tot; f0 += 64 * kAhead)
                        {
                            uint32_t at[kAhead];
                            // A candidate's row: the last one that starts at or
                            // before it.  Where cells are crowded one row holds
                            // all of them, found by two ballots instead of six
                            // dependent LDS reads per candidate (100 k points
                            // in a few cells, another far away, k = 50: 65.7 ->
                            // 29.8 ms per call, 39.1 with a heap per lane).
                            const uint32_t row0 = (uint32_t)__popcll(__ballot(first <= f0));
                            if (row0 == (uint32_t)__popcll(__ballot(first < min(f0 + 64u * kAhead, tot))))
                            {
                                const uint32_t o = readlane(off, row0 - 1u);
#pragma unroll
                                for (uint32_t u = 0; u < kAhead; ++u) at[u] = min(f0 + u * 64u + lane, tot - 1u) + o;
                            }
                            else
                            {
#pragma unroll
                                for (uint32_t u = 0; u < kAhead; ++u)
                                {
                                    const uint32_t f = min(f0 + u * 64u + lane, tot - 1u);
                                    uint32_t rw = 0;
#pragma unroll
                                    for (uint32_t step = 32; step; step >>= 1)
                                        rw = f >= from_lane(first, rw + step) ? rw + step : rw;
                                    at[u] = f + from_lane(off, rw);
                                }
                            }
                            float4 p[kAhead];
#pragma unroll
                            for (uint32_t u = 0; u < kAhead; ++u) p[u] = gload(pts, at[u]);
                            __builtin_amdgcn_sched_barrier(0);  // (all of them before the first is used)
#pragma unroll
                            for (uint32_t u = 0; u < kAhead; ++u)
                            {
                                const uint32_t d = min(__float_as_uint(sqdist32(qxf, qyf, qzf, p[u].x, p[u].y, p[u].z)), kNanBits);
                                const uint32_t id = __float_as_uint(p[u].w);
                                bool in = (f0 + u * 64u + lane < tot) & (d <= tau);
                                if (tie != 0xFFFFFFFFu) in &= (d < tau) | (id <= tie);
                                const uint64_t m = __ballot(in);
                                if (in) buf[n_buf + lanes_below(m)] = ((uint64_t)d << 32) | id;
                                n_buf = uniform(n_buf + (uint32_t)__popcll(m));
                            }
                            if (n_buf > kBufKeys - 64u * kAhead)
                            {
                                reduce();
                                // k points lie within the new tau: with much
                                // of the old ball left, start over with it
                                again = 2.0f * __uint_as_float(tau) < w && (r0 + 64 < nr || tot - f0 > 1024u);
                                if (again) break;
                            }
                        }
                    }
                    if (again) continue;
                    if (n_buf > kMost) reduce();
                    n = n_buf;
                    if (n >= k || tau >= limit) break;
                    // the next ball: the part of the radius past the grid's
                    // box grows, by the points found (about with its square)
                    const double f = n ? sqrt(fmin(fmax(1.2 * (double)target / (double)n, 1.5), 8.0)) : 2.8;
                    const double past = fmax(sqrt((double)w) - away, 0.25 * h) * f + away;
                    const uint32_t t = uniform(__float_as_uint((float)(past * past)));
                    tau = min(t < 0x7F800000u ? max(t, tau + 1u) : kNanBits, limit);
                    tie = 0xFFFFFFFFu;
                }
                wave_sync();
                for (uint32_t e = lane; e < n; e += 64) row[e] = buf[e];
                wave_sync();
            }
            guess = uniform(__float_as_uint(__uint_as_float(tau) * target * __builtin_amdgcn_rcpf((float)n)));
            n_kept = lane == s ? n : n_kept;
        }

        // ---- the batch's rows, sorted and written ----
        wave_sync();
        {
            const uint32_t q = lane / G, g = (lane % G) * kPerLane;
            const uint32_t n = from_lane(n_kept, q);
            uint64_t* row = kept + q * kStride + g;
            double v[kPerLane];
#pragma unroll
            for (int r = 0; r < kPerLane; ++r)
                v[r] = __longlong_as_double((long long)(g + (uint32_t)r < n ? row[r] : kNoKey));
            sort_rows<G>(v, lane);
#pragma unroll
            for (int r = 0; r < kPerLane; ++r) row[r] = (uint64_t)__double_as_longlong(v[r]);
        }
        wave_sync();
        write_rows(base, nb, kStride, n_kept);
        wave_sync();
    }

    if constexpr (MODE == kModeKnnFeat)
    {
        // ---- features, one query per lane: its row read back (written by
        // this wave), the coordinates gathered from the caller's points four
        // at a time, the next four issued before the current ones are
        // accumulated ----
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        if (lane >= nq) return;
        // this wave's share of the CSR row offsets
        a.out_ptr[t0 + lane] = (t0 + lane) * k;
        if (t0 + lane == a.n_query - 1) a.out_ptr[a.n_query] = a.n_query * k;
        float f[11];
        if ((finite >> lane) & 1ull)
        {
            const uint32_t* row = a.out_idx + (size_t)__float_as_uint(qv.w) * k;
            const float3* __restrict__ xyz3 = reinterpret_cast<const float3*>(a.data);
            Moments m;
            mom_zero(m);
            constexpr uint32_t kChunk = 4;
            float3 pn[kChunk];
#pragma unroll
            for (uint32_t u = 0; u < kChunk; ++u) pn[u] = xyz3[row[u < k ? u : 0]];
            const double ox = pn[0].x, oy = pn[0].y, oz = pn[0].z;
            for (uint32_t j0 = 0; j0 < k; j0 += kChunk)
            {
                float3 pc[kChunk];
#pragma unroll
                for (uint32_t u = 0; u < kChunk; ++u) pc[u] = pn[u];
                if (j0 + kChunk < k)
                {
#pragma unroll
                    for (uint32_t u = 0; u < kChunk; ++u)
                    {
                        const uint32_t j = j0 + kChunk + u;
                        pn[u] = xyz3[row[j < k ? j : 0]];
                    }
                }
#pragma unroll
                for (uint32_t u = 0; u < kChunk; ++u)
                    if (j0 + u < k) mom_add(m, (double)pc[u].x - ox, (double)pc[u].y - oy, (double)pc[u].z - oz);
            }
            double c[6];
            mom_cov(m, (double)k, c);
            const Eig E = eig_full(c);
            const Pca32 P = to_pca32(E);
            features11(P, f);
        }
        else
            for (int c = 0; c < 11; ++c) f[c] = 0.0f;
        store_row11(a.out_feat + (size_t)__float_as_uint(qv.w) * 11, f);
    }
}

template <int G, int WAVES>
hipError_t launch_wave_w(int mode, uint32_t nb, const WaveArgs& a, hipStream_t s)
{
    if (mode == kModeKnn)
        k_wave_search<kModeKnn, G, WAVES><<<nb, 64, 0, s>>>(a);
    else if (mode == kModeKnnFeat)
        k_wave_search<kModeKnnFeat, G, WAVES><<<nb, 64, 0, s>>>(a);
    else if constexpr (G >= 4)
    {
        if (mode == kModeRadius)
            k_wave_search<kModeRadius, G, WAVES><<<nb, 64, 0, s>>>(a);
        else
            k_wave_search<kModeRadiusCsr, G, WAVES><<<nb, 64, 0, s>>>(a);
    }
    return hipGetLastError();
}

template <int G>
hipError_t launch_wave_g(int mode, const WaveArgs& a, hipStream_t s)
{
    const bool radius = mode == kModeRadius || mode == kModeRadiusCsr;
    const uint32_t nb = radius ? (a.n_query + 63) / 64 * (64 / a.q_per_wave) : (a.n_query + a.q_per_wave - 1) / a.q_per_wave;
    if constexpr (G == 2)
        if (nb > 4u * 1024u) return launch_wave_w<G, 4>(mode, nb, a, s);  // (1024 SIMDs)
    return launch_wave_w<G, 3>(mode, nb, a, s);
}

}  // namespace

hipError_t launch_wave_search(int mode, const WaveArgs& a, hipStream_t s)
{
    static const char* names[4] = {"knn_search", "radius_search", "knn_features_fused", "radius_search_csr"};
    if (a.n_query == 0) return hipSuccess;
    if (mode < 0 || mode > 3 || a.k < 1 || a.k > kWaveMaxK || a.q_per_wave < 1 || a.q_per_wave > 64 ||
        ((mode & 1) && 64 % a.q_per_wave))
        return hipErrorInvalidValue;
    ProfScope ps(names[mode], s);
    // rows of up to 16 G kept candidates, at least about a fifth more than k:
    // a narrower margin takes more steps to find a threshold (k = 9, 10 and 12
    // by G = 1 / 2, us per call: 10 M uniform points 4836, 5068, 5290 / 4619,
    // 4721, 4711; 10 M LiDAR points 5640, 5755, 6059 / 5513, 5551, 5696; k = 8
    // and fewer within 2 % either way)
    // (radius searches hold a whole ball in their region, 12 groups of 64
    // points rather than 6: 700 k uniform points, 63 hits, cap 24: 1034 us per
    // call with G = 2)
    const bool radius = mode & 1;
    if (!radius && a.k <= 8) return launch_wave_g<1>(mode, a, s);
    if (!radius && a.k <= 27) return launch_wave_g<2>(mode, a, s);
    if (a.k <= 54) return launch_wave_g<4>(mode, a, s);
    return launch_wave_g<8>(mode, a, s);
}

}  // namespace pgeof_amd
