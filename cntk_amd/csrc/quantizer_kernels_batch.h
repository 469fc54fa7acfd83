// gfx950 kernels of the per-column gradient quantizer: whole gradient sets in one launch.
#pragma once

#include "quantizer_kernels_column.h"
#include "quantizer_kernels_short.h"
#include "quantizer_kernels_lanes.h"
#include "quantizer_kernels_register.h"
#include "quantizer_kernels_unquantize.h"

namespace cntkq {

// largest e with begins[e] <= b (begins ascending, begins[0] = 0); b and everything derived from it is uniform over the
// workgroup. One round trip to the table instead of log2(count) dependent ones: the 64 lanes of a wavefront test one
// entry each, and the number of entries <= b, minus one, is the answer; above 64 entries a first pass over every
// stride-th entry narrows the range to at most 64 (4096 entries: two round trips). Every wavefront of the workgroup
// does the same look-up. A workgroup of a batched launch lives a few microseconds, of which the dependent loads of a
// binary search were a noticeable part (8 stripe views of 2048 x 1163 decoded in 15.8 us against 12.2 us for the
// plain launch on the whole matrix).
__device__ __forceinline__ uint32_t batch_find(const uint32_t* __restrict__ begins, uint32_t count, uint32_t b)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t first = 0, n = count;
    while (n > 64)
    {
        const uint32_t stride = (n + 63) / 64;
        const uint32_t idx = lane * stride;
        const uint32_t v = idx < n ? begins[first + idx] : 0xFFFFFFFFu;
        const uint32_t cell = (uint32_t) __popcll(__ballot(v <= b)) - 1u;
        first += cell * stride;
        n = min(stride, n - cell * stride);
    }
    const uint32_t v = lane < n ? begins[first + lane] : 0xFFFFFFFFu;
    return first + (uint32_t) __popcll(__ballot(v <= b)) - 1u;
}

// The value of x, the same for the whole wavefront, but unknown to the compiler: what a body loads through it is loaded there. Recognised as
// the same for several bodies, an entry's fields are all loaded before the first branch, and kernels of many bodies have more of them
// than scalar registers, which every workgroup then pays for.
__device__ __forceinline__ uint32_t opaque_scalar(uint32_t x)
{
    asm volatile("" : "+s"(x));
    return x;
}

// Many matrices in one launch: the workgroups of all matrices form one grid; `begins` (count + 1 entries, ascending)
// gives the first workgroup of every matrix. A matrix is a run of column tiles (quantize_tile_body) or of single columns
// (quantize_colg_body). Removes the per-launch floor (several microseconds) that dominates gradient sets made of many
// small matrices.
struct QuantizeBatchEntry
{
    const float* g;
    const float* r_in;
    float* r_out;
    char* q;
    // 0: tiles (t), 1: columns (c), 2 / 3 / 4: 1-bit columns of 1024 / 2048 / 4096 rows (the unrolled body; c.qcol),
    // 5: columns staged in the residual's memory instead of LDS (c), 6 / 7: columns in registers, up to 3 / 6 pieces per
    // thread (r; below 32 bits); 8 / 9 / 10: members of the register grids (quantize_reg_batch_kernel), up to 4 / 8 / 15 pieces
    // for each of 256 threads, up to 3 / 4 / 6 for each of 1024 (r);
    // 11: columns of at most 16 rows, one thread each (s); 14: short columns, a few lanes each (l)
    uint32_t kind;
    uint32_t pad;
    union // the geometry of the entry's kind
    {
        TileGeom t;
        ColGeom c;
        RegGeom r;
        ShortGeom s;
        LanesGeom l;
    };
    uint32_t reserved[6]; // (keeps the entry at the size the no-allocation call's fixed array is laid out for)
};

template <int NBITS, bool ZT>
__global__ __launch_bounds__(kTileThreads) CNTKQ_SGPRS_FOR_8_WAVES void quantize_batch_kernel(const QuantizeBatchEntry* __restrict__ entries,
                                                                      const uint32_t* __restrict__ begins, uint32_t count)
{
    extern __shared__ f32x4 smem_v4[];
    const uint32_t e = batch_find(begins, count, blockIdx.x);
    const uint32_t index = blockIdx.x - begins[e];
    // geometry by value: read once, then held in registers whatever the kernel stores
    if (entries[e].kind == 0)
    {
        const TileGeom t = entries[e].t;
        quantize_tile_body<NBITS, ZT>(entries[e].g, entries[e].r_in, entries[e].r_out, entries[e].q, t, index);
    }
    else if (entries[e].kind == 11)
    {
        const ShortGeom t = entries[e].s;
        quantize_short_body<NBITS, ZT>(entries[e].g, entries[e].r_in, entries[e].r_out, entries[e].q, t, index, reinterpret_cast<float*>(smem_v4));
    }
    else if (NBITS < 32 && entries[e].kind == 14)
    {
        if constexpr (NBITS < 32)
        {
            // (By value the geometry has the other bodies move a dozen scalars to a vector register and back once per column: 26 at 1 bit, 14 to 16 at
            // more. By reference they are 8 and 0, and 48 sets 0.24 % slower, at 1 bit 0.43 %; the stripes' 47 and 12, and level.)
            const QuantizeBatchEntry& en = entries[opaque_scalar(e)];
            const LanesGeom t = en.l;
            quantize_lanes_any<NBITS, ZT, float>(en.g, en.r_in, en.r_out, en.q, t, index, reinterpret_cast<char*>(smem_v4));
        }
    }
    else if (entries[e].kind == 5)
    {
        const ColGeom c = entries[e].c;
        quantize_colg_body<NBITS, ZT, true>(entries[e].g, entries[e].r_in, entries[e].r_out, entries[e].q, c, index, smem_v4);
    }
    else if (NBITS < 32 && entries[e].kind >= 6) // (6 or 7)
    {
        // the column in registers: the bytes of the LDS column body, a fifth faster from 2304 rows up
        if constexpr (NBITS < 32)
        {
            const RegGeom c = entries[e].r;
            if (entries[e].kind == 6)
                quantize_reg_body<NBITS, ZT, kTileThreads, 3>(entries[e].g, entries[e].r_in, entries[e].r_out, entries[e].q, c, index, smem_v4);
            else
                quantize_reg_body<NBITS, ZT, kTileThreads, 6>(entries[e].g, entries[e].r_in, entries[e].r_out, entries[e].q, c, index, smem_v4);
        }
    }
    else if (NBITS != 1 || entries[e].kind == 1)
    {
        const ColGeom c = entries[e].c;
        quantize_colg_body<NBITS, ZT>(entries[e].g, entries[e].r_in, entries[e].r_out, entries[e].q, c, index, smem_v4);
    }
    else if constexpr (NBITS == 1)
    {
        // the unrolled 1-bit column bodies: two thirds of the general body's instructions for the same bytes
        const uint64_t qcol = entries[e].c.qcol;
        if (entries[e].kind == 2)
            quantize_col_body<ZT, 1>(entries[e].g, entries[e].r_in, entries[e].r_out, entries[e].q, qcol, index, smem_v4);
        else if (entries[e].kind == 3)
            quantize_col_body<ZT, 2>(entries[e].g, entries[e].r_in, entries[e].r_out, entries[e].q, qcol, index, smem_v4);
        else
            quantize_col_body<ZT, 4>(entries[e].g, entries[e].r_in, entries[e].r_out, entries[e].q, qcol, index, smem_v4);
    }
}

// The members whose columns the plain call keeps in registers with edge elements or on 1024 threads, and columns of whole
// pieces too tall for the grid above to hold in 64 registers: one grid for those on T = 256 threads, one for those on 1024.
// Launched one by one, each such matrix took at least the 4.4 us of a launch, and its last workgroups ran alone on the device:
// a network of 20 matrices at 2 bits (755 to 14336 rows, 4 workers) spent 16 launches and 240 us on them. The body with
// edge elements serves whole columns too (it then has none), so the bytes are the plain call's. A column of few pieces per thread does not
// execute the slots of the taller members: the bodies differ in PER only.
constexpr int kRegBatchPer256[3] = {4, 8, 15};
constexpr int kRegBatchPer1024[3] = {3, 4, 6};

// WIDE (T = 256): also members of more than 8 pieces per thread (five wavefronts per SIMD instead of six)
template <int T, bool WIDE>
constexpr int reg_batch_waves() // (seven for eight pieces would cost a few spilled registers)
{
    return T == 1024 ? 8 : (WIDE ? 5 : 6);
}

template <int NBITS, bool ZT, int T, bool WIDE>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(reg_batch_waves<T, WIDE>(), reg_batch_waves<T, WIDE>()))) void
quantize_reg_batch_kernel(const QuantizeBatchEntry* __restrict__ entries, const uint32_t* __restrict__ begins, uint32_t count)
{
    extern __shared__ f32x4 smem_v4[];
    const uint32_t e = batch_find(begins, count, blockIdx.x);
    const uint32_t column = blockIdx.x - begins[e];
    const QuantizeBatchEntry& en = entries[e];
    const RegGeom c = en.r;
    constexpr const int(&P)[3] = T == 1024 ? kRegBatchPer1024 : kRegBatchPer256;
    if (en.kind == 8)
        quantize_reg_body<NBITS, ZT, T, P[0], true>(en.g, en.r_in, en.r_out, en.q, c, column, smem_v4);
    else if ((T == 256 && !WIDE) || en.kind == 9)
        quantize_reg_body<NBITS, ZT, T, P[1], true>(en.g, en.r_in, en.r_out, en.q, c, column, smem_v4);
    else if constexpr (T == 1024 || WIDE)
        quantize_reg_body<NBITS, ZT, T, P[2], true>(en.g, en.r_in, en.r_out, en.q, c, column, smem_v4);
}

// The owner's stripe reductions of a whole gradient set in one launch: same grid construction as quantize_batch_kernel.
struct StripeBatchEntry
{
    StripeSources src;
    float* stripe_res;
    char* q_out;
    float* agg_out;
    // 0: tiles (t), 1: columns (c), 2 / 3: 1-bit columns of 1024 / 2048 rows (the unrolled body; c.qcol),
    // 4 / 5: 1-bit columns of up to eight workers, sums looked up, up to 3 / 6 pieces per thread (r);
    // 8 / 9 / 10: members of the register grids, pieces as QuantizeBatchEntry has them (r, group);
    // 11: columns of at most 16 rows (s); 12 / 13: columns of a single worker, up to 3 / 6 pieces per thread (r);
    // 14: short columns of a single worker, a few lanes each (l)
    uint32_t kind;
    uint32_t group; // workers whose packed columns are in LDS together
    TileGeom t;
    ColGeom c;
    RegGeom r;
    ShortGeom s;
    LanesGeom l;
};

// LOOKUP: the variant that also runs members of kinds 4 and 5 (76 registers instead of 44: a launch without such members
// takes the other one and keeps eight wavefronts per SIMD)
template <int NBITS, bool ZT, bool LOOKUP>
__device__ __forceinline__ void stripe_reduce_batch_body(const StripeBatchEntry* __restrict__ entries, const uint32_t* __restrict__ begins,
                                                         uint32_t count)
{
    extern __shared__ f32x4 smem_v4[];
    const uint32_t e = batch_find(begins, count, blockIdx.x);
    const uint32_t index = blockIdx.x - begins[e];
    const StripeBatchEntry& en = entries[e]; // the table is read-only while the kernel runs
    if (en.kind == 0)
    {
        const TileGeom t = en.t;
        stripe_reduce_tile_body<NBITS, ZT>(en.src, en.stripe_res, en.q_out, en.agg_out, t, index);
    }
    else if (en.kind == 11)
    {
        const ShortGeom t = en.s;
        stripe_reduce_short_body<NBITS, ZT>(en.src, en.stripe_res, en.q_out, en.agg_out, t, index, reinterpret_cast<float*>(smem_v4));
    }
    else if (NBITS != 1 || en.kind == 1)
    {
        const ColGeom c = en.c;
        stripe_reduce_colg_body<NBITS, ZT>(en.src, en.stripe_res, en.q_out, en.agg_out, c, index, smem_v4);
    }
    else if (LOOKUP && NBITS == 1 && en.kind >= 4)
    {
        // the plain call's kernel for these stripes: the bytes of the general column body, up to twice as fast
        if constexpr (LOOKUP && NBITS == 1)
        {
            const RegGeom c = en.r;
            if (en.kind == 4)
                stripe_reduce_lut_body<ZT, 3, kTileThreads>(en.src, en.stripe_res, en.q_out, en.agg_out, c, index, smem_v4);
            else
                stripe_reduce_lut_body<ZT, 6, kTileThreads>(en.src, en.stripe_res, en.q_out, en.agg_out, c, index, smem_v4);
        }
    }
    else if constexpr (NBITS == 1)
    {
        const uint64_t qcol = en.c.qcol;
        // (workgroups with the same index modulo 8 run on one die wherever the member starts in the grid)
        const uint32_t column = column_of_workgroup(index, begins[e + 1] - begins[e]);
        // (4096 rows stay with the general body: unrolled they take 74 registers, which would cost every member of the
        // launch two of its eight wavefronts per SIMD)
        if (en.kind == 2)
            stripe_reduce_col_body<ZT, 1>(en.src, en.stripe_res, en.q_out, en.agg_out, qcol, column, smem_v4);
        else
            stripe_reduce_col_body<ZT, 2>(en.src, en.stripe_res, en.q_out, en.agg_out, qcol, column, smem_v4);
    }
}

// The stripes of a single worker: columns of up to six pieces per thread as quantize_reg_body has them (kinds 12 / 13: up to 3 / 6
// pieces; r), the rest as above. At 1 bit (a level picked by a bit) six pieces fit 64 registers; a code's decoding takes two more, and
// a wavefront less is cheaper than 20 bytes of scratch (eight wavefronts / seven, us: stripes of 2049 to 6144 rows at 8 bits 32.6 / 31.3,
// ResNet-50 at 2 bits 55.9 / 53.8, at 8 bits 58.9 / 58.4; up to 3072 rows, where the scratch is not touched, at 8 bits 18.7 / 19.0).
constexpr int stripe_one_batch_waves(int nbits)
{
    return nbits == 1 || nbits == 32 ? 8 : 7;
}

template <int NBITS, bool ZT>
__global__ __launch_bounds__(kTileThreads) __attribute__((amdgpu_waves_per_eu(stripe_one_batch_waves(NBITS), stripe_one_batch_waves(NBITS)))) CNTKQ_SGPRS_FOR_8_WAVES void stripe_one_batch_kernel(const StripeBatchEntry* __restrict__ entries,
                                                                                                const uint32_t* __restrict__ begins, uint32_t count)
{
    extern __shared__ f32x4 smem_v4[];
    const uint32_t e = batch_find(begins, count, blockIdx.x);
    const uint32_t index = blockIdx.x - begins[e];
    const StripeBatchEntry& en = entries[e];
    if (en.kind == 0)
    {
        const TileGeom t = en.t;
        stripe_reduce_tile_body<NBITS, ZT>(en.src, en.stripe_res, en.q_out, en.agg_out, t, index);
    }
    else if (en.kind == 11)
    {
        const ShortGeom t = en.s;
        stripe_reduce_short_body<NBITS, ZT>(en.src, en.stripe_res, en.q_out, en.agg_out, t, index, reinterpret_cast<float*>(smem_v4));
    }
    else if (NBITS < 32 && en.kind == 14)
    {
        if constexpr (NBITS < 32)
        {
            const StripeBatchEntry& le = entries[opaque_scalar(e)];
            const LanesGeom t = le.l;
            stripe_lanes_any<NBITS, ZT, float>(le.src, le.stripe_res, le.q_out, le.agg_out, t, index, reinterpret_cast<char*>(smem_v4));
        }
    }
    else if constexpr (NBITS == 32)
    {
        const ColGeom c = en.c;
        stripe_reduce_colg_body<NBITS, ZT>(en.src, en.stripe_res, en.q_out, en.agg_out, c, index, smem_v4);
    }
    else
    {
        const RegGeom c = en.r;
        if (en.kind == 12)
            stripe_one_reg_body<NBITS, ZT, kTileThreads, 3>(en.src.q[0], en.stripe_res, en.q_out, en.agg_out, c, index, smem_v4);
        else
            stripe_one_reg_body<NBITS, ZT, kTileThreads, 6>(en.src.q[0], en.stripe_res, en.q_out, en.agg_out, c, index, smem_v4);
    }
}

template <int NBITS, bool ZT>
__global__ __launch_bounds__(kTileThreads) CNTKQ_SGPRS_FOR_8_WAVES void stripe_reduce_batch_kernel(const StripeBatchEntry* __restrict__ entries,
                                                                                                   const uint32_t* __restrict__ begins, uint32_t count)
{
    stripe_reduce_batch_body<NBITS, ZT, false>(entries, begins, count);
}

// (six wavefronts per SIMD by its vector registers: as many scalar registers as the compiler likes)
template <bool ZT>
__global__ __launch_bounds__(kTileThreads) void stripe_reduce_batch_lookup_kernel(const StripeBatchEntry* __restrict__ entries,
                                                                                  const uint32_t* __restrict__ begins, uint32_t count)
{
    stripe_reduce_batch_body<1, ZT, true>(entries, begins, count);
}

// Stripes whose sums the plain call keeps in registers (with edge elements or on 1024 threads), in one grid per workgroup size:
// see quantize_reg_batch_kernel. 1 bit: up to eight workers, sums looked up; otherwise decoded worker by worker.
template <int NBITS, bool ZT, int T, int PER>
__device__ __forceinline__ void stripe_reduce_reg_member(const StripeBatchEntry& en, const RegGeom& c, uint32_t column, f32x4* smem_v4)
{
    if constexpr (NBITS == 1)
        stripe_reduce_lut_body<ZT, PER, T>(en.src, en.stripe_res, en.q_out, en.agg_out, c, column, smem_v4);
    else
        stripe_reduce_reg_body<NBITS, ZT, PER, T>(en.src, en.stripe_res, en.q_out, en.agg_out, c, en.group, column, smem_v4);
}

template <int NBITS, int T, bool WIDE>
constexpr int stripe_reg_batch_waves()
{
    return T == 1024 ? 8 : (WIDE ? (NBITS == 1 ? 5 : 4) : 7);
}

template <int NBITS, bool ZT, int T, bool WIDE>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(stripe_reg_batch_waves<NBITS, T, WIDE>(), stripe_reg_batch_waves<NBITS, T, WIDE>()))) void
stripe_reduce_reg_batch_kernel(const StripeBatchEntry* __restrict__ entries, const uint32_t* __restrict__ begins, uint32_t count)
{
    extern __shared__ f32x4 smem_v4[];
    const uint32_t e = batch_find(begins, count, blockIdx.x);
    const uint32_t column = blockIdx.x - begins[e];
    const StripeBatchEntry& en = entries[e];
    const RegGeom c = en.r;
    constexpr const int(&P)[3] = T == 1024 ? kRegBatchPer1024 : kRegBatchPer256;
    if (en.kind == 8)
        stripe_reduce_reg_member<NBITS, ZT, T, P[0]>(en, c, column, smem_v4);
    else if ((T == 256 && !WIDE) || en.kind == 9)
        stripe_reduce_reg_member<NBITS, ZT, T, P[1]>(en, c, column, smem_v4);
    else if constexpr (T == 1024 || WIDE)
        stripe_reduce_reg_member<NBITS, ZT, T, P[2]>(en, c, column, smem_v4);
}

// ... of a single worker (WIDE: fifteen pieces take seven registers more than four wavefronts per SIMD leave; three without scratch
// memory against four with it: stripes of 8200 to 14336 rows at 1 / 8 bits 17.6 / 19.1 -> 17.0 / 17.2 us)
template <int T, bool WIDE>
constexpr int stripe_one_reg_batch_waves()
{
    return T == 1024 ? 8 : (WIDE ? 3 : 6);
}

template <int NBITS, bool ZT, int T, bool WIDE>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(stripe_one_reg_batch_waves<T, WIDE>(), stripe_one_reg_batch_waves<T, WIDE>()))) void
stripe_one_reg_batch_kernel(const StripeBatchEntry* __restrict__ entries, const uint32_t* __restrict__ begins, uint32_t count)
{
    extern __shared__ f32x4 smem_v4[];
    const uint32_t e = batch_find(begins, count, blockIdx.x);
    const uint32_t column = blockIdx.x - begins[e];
    const StripeBatchEntry& en = entries[e];
    const RegGeom c = en.r;
    constexpr const int(&P)[3] = T == 1024 ? kRegBatchPer1024 : kRegBatchPer256;
    if (en.kind == 8)
        stripe_one_reg_body<NBITS, ZT, T, P[0]>(en.src.q[0], en.stripe_res, en.q_out, en.agg_out, c, column, smem_v4);
    else if ((T == 256 && !WIDE) || en.kind == 9)
        stripe_one_reg_body<NBITS, ZT, T, P[1]>(en.src.q[0], en.stripe_res, en.q_out, en.agg_out, c, column, smem_v4);
    else if constexpr (T == 1024 || WIDE)
        stripe_one_reg_body<NBITS, ZT, T, P[2]>(en.src.q[0], en.stripe_res, en.q_out, en.agg_out, c, column, smem_v4);
}

// Many matrices in one launch (see quantize_batch_kernel): the 256-thread blocks of all matrices form one grid.
enum UnqKind : uint32_t
{
    kUnqVec4 = 0,    // QWord-major, 16-byte stores
    kUnqScalar = 1,  // QWord-major, 4-byte stores
    kUnqSegment = 2, // segment decoder
    kUnqRows = 3,    // row-major decoder, packed column in LDS
    kUnqTile = 4,    // several short columns per workgroup, packed records in LDS
    kUnqDirect = 5,  // row-major decoder, QWords fetched by the threads that decode them (geometry in rowg)
    kUnqFlat = 6     // the same for short columns: the matrix as one run of groups of consecutive elements
};

struct UnquantizeBatchEntry
{
    const char* q;
    float* out;
    uint32_t kind;
    uint32_t pad;
    UnqGeom qw;      // valid for kUnqVec4 / kUnqScalar
    UnqSegGeom seg;  // valid for kUnqSegment
    UnqRowGeom rowg; // valid for kUnqRows / kUnqDirect
    UnqTileGeom tile; // valid for kUnqTile
    UnqFlatGeom flat; // valid for kUnqFlat
};

template <int NBITS>
__global__ __launch_bounds__(256) void unquantize_batch_kernel(const UnquantizeBatchEntry* __restrict__ entries,
                                                               const uint32_t* __restrict__ begins, uint32_t count, int add)
{
    extern __shared__ f32x4 smem_v4[];
    const uint32_t e = batch_find(begins, count, blockIdx.x);
    const UnquantizeBatchEntry& en = entries[e];
    const uint32_t block = blockIdx.x - begins[e];
    if (en.kind == kUnqVec4)
        unquantize_body<NBITS, 4>(en.q, en.out, en.qw, add, block);
    else if (en.kind == kUnqScalar)
        unquantize_body<NBITS, 1>(en.q, en.out, en.qw, add, block);
    else if (en.kind == kUnqSegment)
        unquantize_segment_body<NBITS>(en.q, en.out, en.seg, add, block);
    else if (en.kind == kUnqRows)
    {
        const UnqRowGeom t = en.rowg; // by value: the loop below stores between its uses
        unquantize_rows_body<NBITS>(en.q, en.out, t, add, block, reinterpret_cast<uint32_t*>(smem_v4));
    }
    else if (en.kind == kUnqDirect)
    {
        const UnqRowGeom t = en.rowg;
        unquantize_direct_body<NBITS>(en.q, en.out, t, add, block);
    }
    else if (en.kind == kUnqFlat)
    {
        const UnqFlatGeom t = en.flat;
        unquantize_flat_body<NBITS>(en.q, en.out, t, add, block);
    }
    else
    {
        const UnqTileGeom t = en.tile;
        unquantize_tile_body<NBITS>(en.q, en.out, t, add, block, reinterpret_cast<uint32_t*>(smem_v4));
    }
}

} // namespace cntkq
