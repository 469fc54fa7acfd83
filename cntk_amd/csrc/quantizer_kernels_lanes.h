// gfx950 kernels of the per-column gradient quantizer: short columns, a few to a wavefront, for quantize and for the stripe
// reduction, both element types.
#pragma once

#include "quantizer_kernels_tile.h"     // StripeSources, stripe_order, lds_or
#include "quantizer_kernels_strip.h"    // StripElem
#include "quantizer_kernels_register.h" // opaque

namespace cntkq {

// A wavefront takes 64 / lanes consecutive columns, one run of memory. Gradient + residual go to its own part of LDS in 16-byte pieces,
// each lane takes its share of a column into registers -- elements l, l + lanes, ... for lane l, at most 20 (CHAIN) -- and statistics, codes and
// residual are worked out from there; the residual and the records, bounds and QWords, leave LDS as one run each.
// These are the tile kernels' steps, sums and bytes, a lane for each of their threads per column. What is different: nothing crosses
// a wavefront, so there is no barrier and no wavefront waits for another one's loads, all of a wavefront's loads are in flight together, and
// a value is read out of LDS once instead of three times. What bounds a small matrix is the length of one wavefront's chain of
// latencies (memory, LDS, the butterflies and divisions of the bounds), a large one memory. Tile kernel / this at 1 bit, us a launch among others:
// 512 rows 6.5 / 4.6 at 100000 elements, 7.1 / 5.4 at 1 M, 25.3 / 22.3 (4.8 / 5.4 TB/s) at 10 M; 147 rows 7.7 / 5.0, 8.9 / 6.1 and 25.7 / 23.9;
// 1023 rows 7.1 / 5.3, 7.8 / 6.0 and 26.2 / 25.2; 32 rows 4.5 / 3.3, 7.6 / 4.8 and 45.5 / 24.8.
constexpr uint32_t kLanesThreads = 256;
constexpr uint32_t kLanesWaves = kLanesThreads / 64;
constexpr uint32_t kLanesMaxChain = 20;

struct LanesGeom
{
    uint32_t rows;
    uint32_t cols;
    uint32_t nq;
    uint32_t lanes;      // lanes per column: 8, 16, 32 or 64
    uint32_t lanes_log2;
    uint32_t chain;      // elements per lane the kernel is instantiated for: 4, 8, 16 or 20
    uint32_t step_k;     // lanes / nq and
    uint32_t step_w;     // lanes % nq: how far a lane's next element lies in bit positions and QWords
    uint32_t run_elems;  // elements of LDS for a wavefront's columns, whole 16-byte pieces
    uint32_t rec_words;  // QWords of LDS for its records, whole 16-byte pieces
    uint64_t qcol;
};

// workers: 0 for a quantize call; the reduction keeps what decodes a worker's codes, two values per worker and column
template <typename E>
__host__ __device__ inline uint32_t lanes_wave_elems(const LanesGeom& t, uint32_t workers)
{
    return t.run_elems + t.rec_words + (((64u >> t.lanes_log2) * 2 * workers + 3u) & ~3u);
}
template <typename E>
inline size_t lanes_lds_bytes(const LanesGeom& t, size_t workers)
{
    return (size_t) kLanesWaves * lanes_wave_elems<E>(t, (uint32_t) workers) * sizeof(E);
}

// orders what the lanes of a wavefront have written to LDS before what they read from it afterwards
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// lanes_sum without branches: sums of independent values overlap
template <typename T>
__device__ __forceinline__ T group_sum_any(T v, uint32_t lanes)
{
    v += dpp_lane<kDppXor1>(v);
    v += dpp_lane<kDppXor2>(v);
    v += dpp_lane<kDppHalfMirror>(v);
    const T row = v + dpp_lane<kDppMirror>(v);
    T t = row + dpp_lane<kDppBcast15>(row);
    const T half = (threadIdx.x & 32u) ? read_lane(t, 63) : read_lane(t, 31);
    t += dpp_lane<kDppBcast31>(t);
    const T whole = read_lane(t, 63);
    return lanes == 8 ? v : (lanes == 16 ? row : (lanes == 32 ? half : whole));
}

// a column's bounds, at the alignment of an element
template <typename E>
struct LanesPairOf;
template <>
struct LanesPairOf<float>
{
    typedef f32x2_u type;
};
template <>
struct LanesPairOf<double>
{
    typedef f64x2_u type;
};
template <typename E>
using LanesPair = typename LanesPairOf<E>::type;

// A wavefront's part of a matrix: its first column, how many it has, its LDS. (False: the matrix ends before it. A branch, and not a count of
// zero: of `first < cols ? min(per, cols - first) : 0` this compiler makes a saturating subtraction and selects one that is not, on
// scalars, so that wavefronts beyond the last column got a full count.)
template <typename E>
struct LanesWave
{
    uint32_t first, columns;
    E* run;                    // 16-byte aligned
    typename Word<E>::Q* recs; // 16-byte aligned
    E* dec;
};
template <typename E>
__device__ __forceinline__ bool lanes_wave(const LanesGeom& t, uint32_t block, uint32_t workers, char* smem, LanesWave<E>& w)
{
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), per = 64u >> t.lanes_log2;
    w.first = (block * kLanesWaves + wave) * per;
    if (w.first >= t.cols)
        return false;
    w.columns = min(per, t.cols - w.first);
    w.run = reinterpret_cast<E*>(smem) + wave * lanes_wave_elems<E>(t, workers);
    w.recs = reinterpret_cast<typename Word<E>::Q*>(w.run + t.run_elems);
    w.dec = w.run + t.run_elems + t.rec_words;
    return true;
}

// Where a run of `total` elements whose 16-byte phase is that of `at` goes in LDS (the same phase), and how it splits into elements
// before the first aligned piece, pieces, and elements after the last one.
template <typename E>
struct LanesRun
{
    uint32_t mis, head, pieces, tail;
};
template <typename E>
__device__ __forceinline__ LanesRun<E> lanes_run(const E* at, uint32_t total)
{
    constexpr uint32_t N = 16 / sizeof(E);
    LanesRun<E> r;
    r.mis = (uint32_t) (reinterpret_cast<uintptr_t>(at) / sizeof(E)) & (N - 1);
    r.head = min((N - r.mis) & (N - 1), total);
    r.pieces = (total - r.head) / N;
    r.tail = total - r.head - r.pieces * N;
    return r;
}

// run: the wavefront's columns in LDS, one after the other; res: where their residuals go, of the phase `l` describes. recs: their records, the
// QWords zero on entry; qw: where the first one goes.
template <int NBITS, bool ZT, int CHAIN, typename E>
__device__ __forceinline__ void lanes_stats_pack(const LanesWave<E>& wv, E* run, const LanesGeom& t, const LanesRun<E>& l, E* res, char* qw)
{
    using Q = typename Word<E>::Q;
    using SE = StripElem<E>;
    using PS = PackShapeOf<NBITS, Word<E>::kBits>;
    constexpr uint32_t N = SE::PER;
    const uint32_t lane = threadIdx.x % 64, c = lane >> t.lanes_log2, lg = lane & (t.lanes - 1);
    const bool live = c < wv.columns;
    E* column = run + min(c, wv.columns - 1) * t.rows;
    E v[CHAIN];
    // elements that do not exist (dead lanes: whatever)
    const uint32_t missing = (uint32_t) CHAIN - ((t.rows + t.lanes - 1 - lg) >> t.lanes_log2);
#pragma unroll
    for (int u = 0; u < CHAIN; ++u)
    {
        const uint32_t i = lg + (u << t.lanes_log2);
        const bool there = i < t.rows;
        const E x = column[there ? i : 0u];
        v[u] = there ? x : (E) 0; // (an addition of +0 changes no sum)
    }
    E lo, hi;
    if constexpr (NBITS == 1)
    {
        E mean = (E) 0;
        if constexpr (!ZT)
        {
            E s = (E) 0;
#pragma unroll
            for (int u = 0; u < CHAIN; ++u)
                s += v[u];
            mean = group_sum_any(s, t.lanes) / (E) t.rows;
        }
        E s0 = (E) 0, s1 = (E) 0;
        uint32_t n0 = 0;
#pragma unroll
        for (int u = 0; u < CHAIN; ++u)
        {
            const bool below = v[u] < mean;
            s0 += below ? v[u] : (E) 0;
            s1 += below ? (E) 0 : v[u];
            n0 += below ? 1u : 0u;
            // (left alone, the compiler takes the three sums one after the other and keeps a comparison's two scalar registers per element until then)
            asm volatile("" : "+v"(s0), "+v"(s1), "+v"(n0));
        }
        n0 -= (E) 0 < mean ? missing : 0u; // the zeros that stand in for elements that do not exist
        s0 = group_sum_any(s0, t.lanes);
        s1 = group_sum_any(s1, t.lanes);
        n0 = group_sum_any(n0, t.lanes);
        finish_stats_1bit<ZT>(mean, s0, s1, n0, t.rows - n0, t.rows, lo, hi);
    }
    else
    {
        E s = (E) 0;
#pragma unroll
        for (int u = 0; u < CHAIN; ++u)
            s += v[u] * v[u];
        s = group_sum_any(s, t.lanes);
        finish_stats_multibit(s, t.rows, lo, hi);
    }
    const ValueQOf<E> vq = make_vq<NBITS, E>(lo, hi);
    const E val0 = unquantize_value<NBITS, E>(vq, (Q) 0);
    const E val1 = unquantize_value<NBITS, E>(vq, (Q) 1);
    if (live)
    {
        Q* record = wv.recs + c * (t.nq + 2);
        if (lg == 0)
        {
            reinterpret_cast<E*>(record)[0] = lo;
            reinterpret_cast<E*>(record)[1] = hi;
        }
        const uint32_t l0 = opaque(lg);
        uint32_t k = small_div(l0, small_divisor(t.nq));
        uint32_t w = l0 - k * t.nq;
#pragma unroll
        for (int u = 0; u < CHAIN; ++u)
        {
            const uint32_t i = l0 + (u << t.lanes_log2);
            if (i < t.rows)
            {
                const Q code = quantize_value<NBITS, ZT, E>(vq, v[u]);
                E back;
                if constexpr (NBITS == 1)
                    back = code ? val1 : val0;
                else
                    back = unquantize_value<NBITS, E>(vq, code);
                column[i] = v[u] - back;
                lds_or(record + 2 + w, (Q) (code << (k * PS::SHIFT)));
            }
            w += t.step_w;
            k += t.step_k;
            if (w >= t.nq)
            {
                w -= t.nq;
                ++k;
            }
        }
    }
    wave_lds_sync();
    // the residual's phase in LDS is its phase in memory
    for (uint32_t e = lane; e < l.pieces; e += 64)
        __builtin_nontemporal_store(reinterpret_cast<const typename SE::V*>(run + l.head)[e], reinterpret_cast<typename SE::VU*>(res + l.head) + e);
    if (lane < l.head)
        res[lane] = run[lane];
    if (lane < l.tail)
        res[l.head + N * l.pieces + lane] = run[l.head + N * l.pieces + lane];
    Q* to = reinterpret_cast<Q*>(qw);
    for (uint32_t x = lane; x < wv.columns * (t.nq + 2); x += 64)
        to[x] = wv.recs[x];
}

template <int NBITS, bool ZT, int CHAIN, typename E>
__device__ __forceinline__ void quantize_lanes_body(const E* __restrict__ g, const E* r_in, E* r_out, char* __restrict__ q, const LanesGeom& t,
                                                    uint32_t block, char* smem)
{
    static_assert(NBITS < Word<E>::kBits, "whole QWords: nothing to assemble");
    using SE = StripElem<E>;
    constexpr uint32_t N = SE::PER;
    constexpr int FETCH = sizeof(E) == 4 ? 5 : 4; // pieces per lane side by side: all of them (1280 floats, 512 doubles a wavefront)
    LanesWave<E> wv;
    if (!lanes_wave<E>(t, block, 0, smem, wv))
        return;
    const uint32_t lane = threadIdx.x % 64, total = wv.columns * t.rows;
    const size_t base = (size_t) wv.first * t.rows;
    const E* gw = g + base;
    const E* rw = r_in + base;
    const LanesRun<E> l = lanes_run(rw, total);
    E* run = wv.run + l.mis;
    E head = (E) 0, tail = (E) 0;
    const uint32_t tail_at = l.head + N * l.pieces + lane;
    if (lane < l.head)
        head = gw[lane] + rw[lane];
    if (lane < l.tail)
        tail = gw[tail_at] + rw[tail_at];
    for (uint32_t e0 = lane; e0 < l.pieces; e0 += 64 * FETCH)
    {
        typename SE::V a[FETCH], b[FETCH];
#pragma unroll
        for (int u = 0; u < FETCH; ++u)
            if (e0 + 64 * u < l.pieces)
            {
                a[u] = __builtin_nontemporal_load(reinterpret_cast<const typename SE::VU*>(gw + l.head) + e0 + 64 * u);
                b[u] = __builtin_nontemporal_load(reinterpret_cast<const typename SE::VU*>(rw + l.head) + e0 + 64 * u);
            }
#pragma unroll
        for (int u = 0; u < FETCH; ++u)
            if (e0 + 64 * u < l.pieces)
                reinterpret_cast<typename SE::V*>(run + l.head)[e0 + 64 * u] = a[u] + b[u];
    }
    if (lane < l.head)
        run[lane] = head;
    if (lane < l.tail)
        run[tail_at] = tail;
    for (uint32_t x = lane; x < wv.columns * (t.nq + 2); x += 64)
        wv.recs[x] = 0u;
    wave_lds_sync();
    // (the residual output may lie at another phase than the input: the pieces are stored at the alignment of an element)
    lanes_stats_pack<NBITS, ZT, CHAIN, E>(wv, run, t, l, r_out + base, q + (size_t) wv.first * t.qcol);
}

template <int NBITS, bool ZT, int CHAIN, typename E>
__global__ __launch_bounds__(kLanesThreads) void quantize_lanes_kernel(const E* __restrict__ g, const E* r_in, E* r_out, char* __restrict__ q, LanesGeom t)
{
    extern __shared__ f32x4 smem_v4[];
    quantize_lanes_body<NBITS, ZT, CHAIN, E>(g, r_in, r_out, q, t, blockIdx.x, reinterpret_cast<char*>(smem_v4));
}

// Stripe reduction: the stripe residual as one run into LDS, then as the tile kernel decodes: a lane per QWord and eight of its bit positions,
// every worker's QWord in turn, in the fixed order of workers, added to the residual in LDS.
template <int NBITS, bool ZT, int CHAIN, typename E>
__device__ __forceinline__ void stripe_lanes_body(const StripeSources& src, E* stripe_res, char* q_out, E* agg_out, const LanesGeom& t, uint32_t block,
                                                  char* smem)
{
    static_assert(NBITS < Word<E>::kBits, "whole QWords: nothing to assemble");
    using Q = typename Word<E>::Q;
    using SE = StripElem<E>;
    using PS = PackShapeOf<NBITS, Word<E>::kBits>;
    constexpr uint32_t N = SE::PER;
    constexpr int FETCH = sizeof(E) == 4 ? 5 : 4;
    constexpr uint32_t BATCH = sizeof(E) == 4 ? 8 : 4; // QWords fetched together
    const uint32_t K = src.workers;
    LanesWave<E> wv;
    if (!lanes_wave<E>(t, block, K, smem, wv))
        return;
    const uint32_t lane = threadIdx.x % 64, total = wv.columns * t.rows;
    const size_t base = (size_t) wv.first * t.rows, rec_base = (size_t) wv.first * t.qcol;
    E* res = stripe_res + base;
    const LanesRun<E> l = lanes_run(static_cast<const E*>(res), total);
    E* run = wv.run + l.mis;
    const uint32_t tail_at = l.head + N * l.pieces + lane;
    {
        typename SE::V b[FETCH];
        E head = (E) 0, tail = (E) 0;
        if (lane < l.head)
            head = res[lane];
        if (lane < l.tail)
            tail = res[tail_at];
#pragma unroll
        for (int u = 0; u < FETCH; ++u) // (a wavefront's columns are at most 64 * FETCH pieces)
            if (lane + 64 * u < l.pieces)
                b[u] = __builtin_nontemporal_load(reinterpret_cast<const typename SE::VU*>(res + l.head) + lane + 64 * u);
        // the workers' column bounds, in the order of summation (a worker's address is the same for all lanes)
#pragma unroll 1
        for (uint32_t n0 = 0; n0 < K; n0 += BATCH)
        {
            LanesPair<E> h[BATCH];
#pragma unroll
            for (uint32_t j = 0; j < BATCH; ++j)
                if (n0 + j < K && lane < wv.columns)
                    h[j] = *reinterpret_cast<const LanesPair<E>*>(src.q[stripe_order(n0 + j, src.owner)] + rec_base + lane * (uint32_t) t.qcol);
#pragma unroll
            for (uint32_t j = 0; j < BATCH; ++j)
                if (n0 + j < K && lane < wv.columns)
                {
                    wv.dec[2 * (lane * K + n0 + j)] = h[j][0];
                    wv.dec[2 * (lane * K + n0 + j) + 1] = h[j][1];
                }
        }
        for (uint32_t x = lane; x < wv.columns * (t.nq + 2); x += 64)
            wv.recs[x] = 0u;
#pragma unroll
        for (int u = 0; u < FETCH; ++u)
            if (lane + 64 * u < l.pieces)
                reinterpret_cast<typename SE::V*>(run + l.head)[lane + 64 * u] = b[u];
        if (lane < l.head)
            run[lane] = head;
        if (lane < l.tail)
            run[tail_at] = tail;
    }
    wave_lds_sync();
    // ... become what decodes a worker's codes: 1 bit -> the two levels, else (ufactor, lower)
    for (uint32_t x = lane; x < wv.columns * K; x += 64)
    {
        const E lo = wv.dec[2 * x], uf = make_ufactor<NBITS, E>(lo, wv.dec[2 * x + 1]);
        wv.dec[2 * x] = NBITS == 1 ? unquantize_value<NBITS, E>(uf, lo, (Q) 0) : uf;
        wv.dec[2 * x + 1] = NBITS == 1 ? unquantize_value<NBITS, E>(uf, lo, (Q) 1) : lo;
    }
    wave_lds_sync();
    const uint32_t nwords = wv.columns * t.nq;
    const float inv_nwords = small_divisor(nwords), inv_nq = small_divisor(t.nq);
#pragma unroll 1
    for (uint32_t it = lane; it < nwords * PS::CHUNKS; it += 64)
    {
        const uint32_t chunk = PS::CHUNKS == 1 ? 0u : small_div(it, inv_nwords);
        const uint32_t qi = it - chunk * nwords;
        const uint32_t c = small_div(qi, inv_nq);
        const uint32_t w = qi - c * t.nq;
        const uint32_t word_at = c * (uint32_t) t.qcol + (2 + w) * (uint32_t) sizeof(Q);
        const uint32_t sh0 = chunk * PS::SLOTS * PS::SHIFT;
        const E* d = wv.dec + 2 * c * K;
        E acc[PS::SLOTS]; // (x + -0 = x: the first worker's values seed the sums through the same addition as the others)
#pragma unroll
        for (uint32_t kk = 0; kk < PS::SLOTS; ++kk)
            acc[kk] = (E) -0.0;
#pragma unroll 1
        for (uint32_t n0 = 0; n0 < K; n0 += BATCH)
        {
            Q word[BATCH];
#pragma unroll
            for (uint32_t j = 0; j < BATCH; ++j)
                if (n0 + j < K)
                    word[j] = *reinterpret_cast<const Q*>(src.q[stripe_order(n0 + j, src.owner)] + rec_base + word_at);
#pragma unroll
            for (uint32_t j = 0; j < BATCH; ++j)
                if (n0 + j < K)
                {
                    const E d0 = d[2 * (n0 + j)], d1 = d[2 * (n0 + j) + 1];
                    const Q bits = word[j] >> sh0;
#pragma unroll
                    for (uint32_t kk = 0; kk < PS::SLOTS; ++kk)
                    {
                        E x;
                        if constexpr (NBITS == 1 && sizeof(E) == 4)
                            x = pick_level(bits, kk, d0, d1);
                        else if constexpr (NBITS == 1)
                            x = (bits >> kk) & 1u ? d1 : d0;
                        else
                            x = unquantize_value<NBITS, E>(d0, d1, (bits >> (kk * PS::SHIFT)) & PS::CODEMASK);
                        acc[kk] = x + acc[kk];
                    }
                }
        }
        E* column = run + c * t.rows;
        uint32_t i = w + chunk * PS::SLOTS * t.nq;
#pragma unroll
        for (uint32_t kk = 0; kk < PS::SLOTS; ++kk, i += t.nq)
            if (i < t.rows)
            {
                if (agg_out != nullptr)
                    agg_out[base + c * t.rows + i] = acc[kk];
                column[i] = acc[kk] + column[i];
            }
    }
    wave_lds_sync();
    lanes_stats_pack<NBITS, ZT, CHAIN, E>(wv, run, t, l, res, q_out + rec_base);
}

// wavefronts per SIMD the reductions are compiled for
template <typename E>
constexpr int lanes_stripe_waves()
{
    return sizeof(E) == 4 ? 8 : 7;
}

template <int NBITS, bool ZT, int CHAIN, typename E>
__global__ __launch_bounds__(kLanesThreads) __attribute__((amdgpu_waves_per_eu(lanes_stripe_waves<E>(), lanes_stripe_waves<E>())))
CNTKQ_SGPRS_FOR_8_WAVES void stripe_lanes_kernel(StripeSources src, E* stripe_res, char* q_out, E* agg_out, LanesGeom t)
{
    extern __shared__ f32x4 smem_v4[];
    stripe_lanes_body<NBITS, ZT, CHAIN, E>(src, stripe_res, q_out, agg_out, t, blockIdx.x, reinterpret_cast<char*>(smem_v4));
}

// the body of the geometry's chain (the same for the whole workgroup); doubles have at most eight elements per lane
#define CNTKQ_LANES_CHAINS(E, BODY)              \
    if (sizeof(E) == 8 || t.chain <= 8)          \
    {                                            \
        if (t.chain == 4)                        \
            BODY(4)                              \
        else                                     \
            BODY(8)                              \
    }                                            \
    else if constexpr (sizeof(E) == 4)           \
    {                                            \
        if (t.chain == 16)                       \
            BODY(16)                             \
        else                                     \
            BODY(20)                             \
    }
template <int NBITS, bool ZT, typename E>
__device__ __forceinline__ void quantize_lanes_any(const E* __restrict__ g, const E* r_in, E* r_out, char* __restrict__ q, const LanesGeom& t,
                                                   uint32_t block, char* smem)
{
#define CNTKQ_BODY(C) quantize_lanes_body<NBITS, ZT, C, E>(g, r_in, r_out, q, t, block, smem);
    CNTKQ_LANES_CHAINS(E, CNTKQ_BODY)
#undef CNTKQ_BODY
}

template <int NBITS, bool ZT, typename E>
__device__ __forceinline__ void stripe_lanes_any(const StripeSources& src, E* stripe_res, char* q_out, E* agg_out, const LanesGeom& t, uint32_t block,
                                                 char* smem)
{
#define CNTKQ_BODY(C) stripe_lanes_body<NBITS, ZT, C, E>(src, stripe_res, q_out, agg_out, t, block, smem);
    CNTKQ_LANES_CHAINS(E, CNTKQ_BODY)
#undef CNTKQ_BODY
}

} // namespace cntkq
