// gfx950 kernels of the per-column gradient quantizer: columns of at most 16 rows, one thread per column.
#pragma once

#include "quantizer_kernels_tile.h"

namespace cntkq {

// The tile kernels give a column at least 8 threads and a workgroup at most 32 columns, so a workgroup of theirs handles 32 to 512
// values here and lives from its latencies: 1 x 38 M at 4 bits took 1221 us (159 here, 5.7 TB/s), 3 x 4.65 M at 1 bit
// 220 us (37), 12 x 1.37 M 80 us (34, 6.0 TB/s).
// Here a workgroup takes 256 columns or more (about 4096 values): gradient + residual as one run into LDS, 16 bytes
// per access; then every thread takes whole columns out of LDS (a column starts an odd number of elements after the one
// before, so that 64 threads that read their columns' element i meet all banks), works out header, codes and residual, and
// writes the record; the residuals leave as one run.
// The sums are those of the tile kernels to the last bit: element i belongs to the partial sum i % 8, added in ascending order
// from +0, and the eight are added as the butterfly over 8 lanes adds them.
constexpr uint32_t kShortThreads = 256;
constexpr uint32_t kShortMaxRows = 16;
constexpr uint32_t kShortTileBytes = 16 * 1024; // values per workgroup, in bytes, unless 256 columns are more

struct ShortGeom
{
    uint32_t rows;
    uint32_t cols;
    uint32_t nq;
    uint32_t cpt; // columns per workgroup: a multiple of 256
    uint64_t qcol;
};

__host__ __device__ inline uint32_t short_stride(uint32_t rows)
{
    return rows | 1u; // elements from one column to the next in LDS
}

__host__ __device__ inline size_t short_lds_bytes(const ShortGeom& t, size_t element)
{
    return (size_t) t.cpt * short_stride(t.rows) * element;
}

// A run of `total` values between memory and the columns in LDS, 16 bytes at a time at the alignment of a value:
// fetch(u, piece) for four pieces of the run, then place(u, positions in LDS of the piece's pairs, piece); one(position, i) for each
// value after the last whole piece.
template <typename E, typename Fetch, typename Place, typename One>
__device__ __forceinline__ void short_walk(uint32_t total, uint32_t rows, Fetch fetch, Place place, One one)
{
    constexpr uint32_t N = 16 / sizeof(E);
    const uint32_t nvec = total / N;
    const bool padded = (rows & 1u) == 0;
    const float inv = small_divisor(rows);
    for (uint32_t e0 = threadIdx.x; e0 < nvec; e0 += 4 * kShortThreads)
    {
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u)
            if (e0 + u * kShortThreads < nvec)
                fetch(u, e0 + u * kShortThreads);
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u)
        {
            const uint32_t e = e0 + u * kShortThreads;
            if (e < nvec)
            {
                // (values 2 x and 2 x + 1 share a column where columns are padded: those heights are even)
                uint32_t at[N / 2];
#pragma unroll
                for (uint32_t h = 0; h < N / 2; ++h)
                {
                    const uint32_t i = N * e + 2 * h;
                    at[h] = padded ? i + small_div(i, inv) : i;
                }
                place(u, at, e);
            }
        }
    }
    for (uint32_t i = nvec * N + threadIdx.x; i < total; i += kShortThreads)
        one(padded ? i + small_div(i, inv) : i, i);
}

template <typename E>
struct ShortVec
{
    static constexpr uint32_t N = 16 / sizeof(E);
    typedef E Vec __attribute__((ext_vector_type(N)));
    typedef Vec VecAtElem __attribute__((aligned(sizeof(E))));
};

template <typename E>
__device__ __forceinline__ void short_store(const E* tile, E* dst, uint32_t total, uint32_t rows)
{
    using V = ShortVec<E>;
    typename V::VecAtElem* d = reinterpret_cast<typename V::VecAtElem*>(dst);
    short_walk<E>(
        total, rows, [](uint32_t, uint32_t) {},
        [&](uint32_t, const uint32_t(&at)[V::N / 2], uint32_t e) {
            typename V::Vec x;
#pragma unroll
            for (uint32_t h = 0; h < V::N / 2; ++h)
            {
                x[2 * h] = tile[at[h]];
                x[2 * h + 1] = tile[at[h] + 1];
            }
            __builtin_nontemporal_store(x, d + e);
        },
        [&](uint32_t at, uint32_t i) { dst[i] = tile[at]; });
}

// L partial sums (a power of two, the rest of the eight being +0) as the lanes of a wavefront add them
template <uint32_t L, typename T>
__device__ __forceinline__ T short_tree(const T (&p)[L])
{
    if constexpr (L == 1)
        return p[0];
    else if constexpr (L == 2)
        return p[0] + p[1];
    else if constexpr (L == 4)
        return (p[0] + p[1]) + (p[2] + p[3]);
    else
        return ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
}

// Statistics, header, codes and residuals of one column in LDS. RMAX: 2, 4, 8 or 16 >= rows.
template <int NBITS, bool ZT, uint32_t RMAX, typename E>
__device__ __forceinline__ void short_column(E* colv, const ShortGeom& t, char* qc)
{
    typedef typename Word<E>::Q QWord;
    using PS = PackShapeOf<NBITS, Word<E>::kBits>;
    constexpr uint32_t L = RMAX < 8 ? RMAX : 8;
    E v[RMAX];
#pragma unroll
    for (uint32_t i = 0; i < RMAX; ++i)
        v[i] = i < t.rows ? colv[i] : (E) 0;
    E lo, hi;
    if constexpr (NBITS == 1)
    {
        E mean = (E) 0;
        if constexpr (!ZT)
        {
            E p[L];
#pragma unroll
            for (uint32_t l = 0; l < L; ++l)
                p[l] = (E) 0 + v[l];
            if constexpr (RMAX > 8)
            {
#pragma unroll
                for (uint32_t l = 0; l < L; ++l)
                    p[l] = p[l] + v[l + 8]; // (an element past the column adds +0 to a sum that is not -0)
            }
            mean = short_tree<L>(p) / (E) t.rows;
        }
        E p0[L], p1[L];
        uint32_t n0 = 0;
#pragma unroll
        for (uint32_t l = 0; l < L; ++l)
            p0[l] = p1[l] = (E) 0;
#pragma unroll
        for (uint32_t i = 0; i < RMAX; ++i)
        {
            const bool valid = i < t.rows, below = v[i] < mean;
            p0[i % 8 < L ? i % 8 : 0] += valid && below ? v[i] : (E) 0;
            p1[i % 8 < L ? i % 8 : 0] += valid && !below ? v[i] : (E) 0;
            n0 += valid && below ? 1u : 0u;
        }
        finish_stats_1bit<ZT>(mean, short_tree<L>(p0), short_tree<L>(p1), n0, t.rows - n0, t.rows, lo, hi);
    }
    else
    {
        E p[L];
#pragma unroll
        for (uint32_t l = 0; l < L; ++l)
            p[l] = (E) 0 + v[l] * v[l];
        if constexpr (RMAX > 8)
        {
#pragma unroll
            for (uint32_t l = 0; l < L; ++l)
                p[l] = p[l] + v[l + 8] * v[l + 8];
        }
        finish_stats_multibit(short_tree<L>(p), t.rows, lo, hi);
    }
    E* header = reinterpret_cast<E*>(qc);
    header[0] = lo;
    header[1] = hi;
    QWord* bits = reinterpret_cast<QWord*>(qc + 2 * sizeof(E));
    const ValueQOf<E> vq = make_vq<NBITS>(lo, hi);
    const E val0 = unquantize_value<NBITS>(vq, 0u);
    const E val1 = unquantize_value<NBITS>(vq, 1u);
    auto code_of = [&](E x, E& residual) -> QWord {
        const QWord code = quantize_value<NBITS, ZT>(vq, x);
        E back;
        if constexpr (NBITS == 1)
            back = code ? val1 : val0;
        else
            back = unquantize_value<NBITS>(vq, code);
        residual = x - back;
        return code;
    };
    if constexpr (RMAX * NBITS <= (uint32_t) Word<E>::kBits)
    {
        // one QWord: element i is bit position i
        QWord word = 0;
#pragma unroll
        for (uint32_t i = 0; i < RMAX; ++i)
        {
            if (i < t.rows)
            {
                E residual;
                word |= code_of(v[i], residual) << (i * PS::SHIFT);
                colv[i] = residual;
            }
        }
        bits[0] = word;
    }
    else
    {
        for (uint32_t w = 0; w < t.nq; ++w)
        {
            QWord word = 0;
            uint32_t shift = 0;
            for (uint32_t i = w; i < t.rows; i += t.nq)
            {
                E residual;
                word |= code_of(colv[i], residual) << shift;
                colv[i] = residual;
                shift += PS::SHIFT;
            }
            bits[w] = word;
        }
    }
}

template <int NBITS, bool ZT, typename E>
__device__ __forceinline__ void short_columns(E* tile, const ShortGeom& t, uint32_t nc, char* q)
{
    const uint32_t stride = short_stride(t.rows);
    // (the height is the same for the whole matrix: one of the four runs)
    if (t.rows <= 2)
        for (uint32_t c = threadIdx.x; c < nc; c += kShortThreads)
            short_column<NBITS, ZT, 2>(tile + c * stride, t, q + (size_t) c * t.qcol);
    else if (t.rows <= 4)
        for (uint32_t c = threadIdx.x; c < nc; c += kShortThreads)
            short_column<NBITS, ZT, 4>(tile + c * stride, t, q + (size_t) c * t.qcol);
    else if (t.rows <= 8)
        for (uint32_t c = threadIdx.x; c < nc; c += kShortThreads)
            short_column<NBITS, ZT, 8>(tile + c * stride, t, q + (size_t) c * t.qcol);
    else
        for (uint32_t c = threadIdx.x; c < nc; c += kShortThreads)
            short_column<NBITS, ZT, 16>(tile + c * stride, t, q + (size_t) c * t.qcol);
}

template <int NBITS, bool ZT, typename E>
__device__ __forceinline__ void quantize_short_body(const E* __restrict__ g, const E* r_in, E* r_out, char* __restrict__ q, const ShortGeom& t,
                                                    uint32_t block, E* tile)
{
    using V = ShortVec<E>;
    const uint32_t j0 = block * t.cpt;
    const uint32_t nc = min(t.cpt, t.cols - j0);
    const uint32_t total = nc * t.rows;
    const size_t base = (size_t) j0 * t.rows;
    const typename V::VecAtElem* g4 = reinterpret_cast<const typename V::VecAtElem*>(g + base);
    const typename V::VecAtElem* r4 = reinterpret_cast<const typename V::VecAtElem*>(r_in + base);
    typename V::Vec a[4], b[4];
    short_walk<E>(
        total, t.rows,
        [&](uint32_t u, uint32_t e) {
            a[u] = __builtin_nontemporal_load(g4 + e);
            b[u] = __builtin_nontemporal_load(r4 + e);
        },
        [&](uint32_t u, const uint32_t(&at)[V::N / 2], uint32_t) {
#pragma unroll
            for (uint32_t h = 0; h < V::N / 2; ++h)
            {
                tile[at[h]] = a[u][2 * h] + b[u][2 * h];
                tile[at[h] + 1] = a[u][2 * h + 1] + b[u][2 * h + 1];
            }
        },
        [&](uint32_t at, uint32_t i) { tile[at] = g[base + i] + r_in[base + i]; });
    // (the workgroup has read all of its residuals before any is written: r_out may be r_in)
    __syncthreads();
    short_columns<NBITS, ZT>(tile, t, nc, q + (size_t) j0 * t.qcol);
    __syncthreads();
    short_store(tile, r_out + base, total, t.rows);
}

template <int NBITS, bool ZT, typename E>
__global__ __launch_bounds__(kShortThreads) void quantize_short_kernel(const E* __restrict__ g, const E* r_in, E* r_out, char* __restrict__ q,
                                                                       ShortGeom t)
{
    extern __shared__ f32x4 smem_v4[];
    quantize_short_body<NBITS, ZT>(g, r_in, r_out, q, t, blockIdx.x, reinterpret_cast<E*>(smem_v4));
}

// The stripe reduction of the same columns (float): the stripe residual as one run into LDS, the workers' stripes decoded and added
// (owner first, then ascending rank) by the thread that has the column, QWord by QWord, four workers' records in flight.
template <int NBITS>
__device__ __forceinline__ void short_sum_column(const StripeSources& src, float* colv, float* agg_col, const ShortGeom& t, size_t rec)
{
    using PS = PackShape<NBITS>;
    constexpr uint32_t SLOTS = 32 / NBITS < kShortMaxRows ? 32 / NBITS : kShortMaxRows; // values of a QWord that a short column has at most
    constexpr uint32_t BATCH = 4; // (more would cost the set's launch, of which this is one body, a wavefront per SIMD)
    const uint32_t K = src.workers;
    for (uint32_t w = 0; w < t.nq; ++w)
    {
        float acc[SLOTS];
        for (uint32_t n0 = 0; n0 < K; n0 += BATCH)
        {
            uint32_t word[BATCH];
            f32x2 head[BATCH];
#pragma unroll
            for (uint32_t u = 0; u < BATCH; ++u)
                if (n0 + u < K)
                {
                    const char* qc = src.q[stripe_order(n0 + u, src.owner)] + rec;
                    head[u] = *reinterpret_cast<const f32x2_u*>(qc);
                    word[u] = reinterpret_cast<const uint32_t*>(qc + 8)[w];
                }
#pragma unroll
            for (uint32_t u = 0; u < BATCH; ++u)
                if (n0 + u < K)
                {
                    const float lo = head[u].x;
                    const float uf = make_ufactor<NBITS>(lo, head[u].y);
                    const float val0 = unquantize_value<NBITS>(uf, lo, 0u);
                    const float val1 = unquantize_value<NBITS>(uf, lo, 1u);
#pragma unroll
                    for (uint32_t k = 0; k < SLOTS; ++k)
                    {
                        float x;
                        if constexpr (NBITS == 1)
                            x = pick_level(word[u], k, val0, val1);
                        else
                            x = unquantize_value<NBITS>(uf, lo, (word[u] >> (k * PS::SHIFT)) & PS::CODEMASK);
                        // the first term seeds the sum; afterwards: decoded value + running sum
                        acc[k] = n0 + u == 0 ? x : x + acc[k];
                    }
                }
        }
#pragma unroll
        for (uint32_t k = 0; k < SLOTS; ++k)
        {
            const uint32_t i = w + k * t.nq;
            if (i < t.rows)
            {
                if (agg_col != nullptr)
                    agg_col[i] = acc[k];
                colv[i] = acc[k] + colv[i];
            }
        }
    }
}

template <int NBITS, bool ZT>
__device__ __forceinline__ void stripe_reduce_short_body(const StripeSources& src, float* stripe_res, char* q_out, float* agg_out, const ShortGeom& t,
                                                         uint32_t block, float* tile)
{
    const uint32_t j0 = block * t.cpt;
    const uint32_t nc = min(t.cpt, t.cols - j0);
    const uint32_t total = nc * t.rows;
    const size_t base = (size_t) j0 * t.rows;
    const uint32_t stride = short_stride(t.rows);
    float* sp = stripe_res + base;
    const f32x4_u* s4 = reinterpret_cast<const f32x4_u*>(sp);
    f32x4 a[4];
    short_walk<float>(
        total, t.rows, [&](uint32_t u, uint32_t e) { a[u] = __builtin_nontemporal_load(s4 + e); },
        [&](uint32_t u, const uint32_t(&at)[2], uint32_t) {
            tile[at[0]] = a[u].x;
            tile[at[0] + 1] = a[u].y;
            tile[at[1]] = a[u].z;
            tile[at[1] + 1] = a[u].w;
        },
        [&](uint32_t at, uint32_t i) { tile[at] = sp[i]; });
    __syncthreads();
    // (a thread reads every worker's record of a column before it writes that column's: q_out may be the owner's stripe)
    for (uint32_t c = threadIdx.x; c < nc; c += kShortThreads)
        short_sum_column<NBITS>(src, tile + c * stride, agg_out != nullptr ? agg_out + base + (size_t) c * t.rows : nullptr, t,
                                (size_t) (j0 + c) * t.qcol);
    short_columns<NBITS, ZT>(tile, t, nc, q_out + (size_t) j0 * t.qcol);
    __syncthreads();
    short_store(tile, sp, total, t.rows);
}

template <int NBITS, bool ZT>
__global__ __launch_bounds__(kShortThreads) CNTKQ_SGPRS_FOR_8_WAVES void stripe_reduce_short_kernel(StripeSources src, float* stripe_res, char* q_out,
                                                                                                    float* agg_out, ShortGeom t)
{
    extern __shared__ f32x4 smem_v4[];
    stripe_reduce_short_body<NBITS, ZT>(src, stripe_res, q_out, agg_out, t, blockIdx.x, reinterpret_cast<float*>(smem_v4));
}

} // namespace cntkq
