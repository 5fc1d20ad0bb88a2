// What the fp32 GEMM's translation units share: a launch's arguments, the order in which its
// workgroups take tiles, and what is stored for a sum.
#ifndef SPH_GEMM_F32_H
#define SPH_GEMM_F32_H

#include "sph_internal.h"

namespace sph
{
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
// four floats that need only be 4-byte aligned: the rows of out start anywhere when N is no
// multiple of 4, and a 16-byte vector memory access only asks for dword alignment
typedef floatx4 floatx4a4 __attribute__((aligned(4)));

struct GemmF32Args
{
    float* out;
    const float* A;
    const float* B;
    const SphGemmEntry* entries;  // device table, or null for stride arithmetic
    uint32_t M, N, K;
    // floats between consecutive rows of B as stored K x N and of out: N, unless a launch covers
    // some of the columns of a wider matrix; likewise of an A stored K x M: M, unless a launch
    // covers some of the rows
    uint32_t ldb, ldc, lda;
    uint32_t split;      // launcher: 1 = a part of the columns, 2 = a part of the rows, 4 = the
                         // tiled kernels have been chosen, 8 = the K-split kernel among them,
                         // 16 = a thin strip of a wider product: the few-tile kernel, 16 x 16
                         // tiles, four wavefronts
    uint32_t basesOk;    // launcher: the caller's A and B start on 16-byte boundaries
    uint32_t tilesM, tilesN;
    uint32_t tilesTotal;  // tilesM * tilesN * units
    uint32_t perXcd;      // ceil(tilesTotal / 8): the grid has 8 * perXcd workgroups
    uint32_t band;        // tile rows per band of the in-unit ordering
    uint32_t overwrite;  // out = A*B instead of out += A*B
    uint32_t relu;       // out = max(., 0) applied to the value that is stored
    const float* bias;   // when set: out = (0 + bias[column]) + A*B, out is not read
    // when sgd is set: out = out - ((A*B) * sgdScale) * sgdRate, every operation rounded on its
    // own -- the update Scale + Sub apply to a gradient that was stored first
    uint32_t sgd;
    uint32_t mirror;     // launcher, few columns: operands, M and N changed places, out did not
    float sgdScale, sgdRate;
    int64_t strideOut, strideA, strideB;
};

// Workgroup -> tile.  Workgroups are handed to the 8 XCDs round robin (id % 8), and each XCD
// has its own L2.  Workgroup `id` therefore takes logical tile (id % 8) * perXcd + id / 8, so
// that an XCD owns one contiguous run of logical tiles; inside a unit the logical order walks
// bands of `band` tile rows column by column, which makes a run a compact block of the
// output whose A rows and B columns the XCD's workgroups share.  Returns false for the
// surplus workgroups of a grid rounded up to 8 * perXcd.
__device__ __forceinline__ void MapLogical(const GemmF32Args& args, uint32_t logical, uint32_t& tm,
                                           uint32_t& tn, uint32_t& unit)
{
    const uint32_t perUnit = args.tilesM * args.tilesN;
    unit = logical / perUnit;
    const uint32_t t = logical - unit * perUnit;
    const uint32_t perBand = args.band * args.tilesN;
    const uint32_t bandIdx = t / perBand;
    const uint32_t within = t - bandIdx * perBand;
    const uint32_t rows = min(args.band, args.tilesM - bandIdx * args.band);
    tm = bandIdx * args.band + within % rows;
    tn = within / rows;
}

__device__ __forceinline__ bool MapTile(const GemmF32Args& args, uint32_t& tm, uint32_t& tn,
                                        uint32_t& unit)
{
    const uint32_t id = blockIdx.x;
    const uint32_t logical = (id & 7u) * args.perXcd + (id >> 3);
    if (logical >= args.tilesTotal)
        return false;
    MapLogical(args, logical, tm, tn, unit);
    return true;
}

// What is stored for an element whose old value (or bias term) is `old` and whose product sum
// is `sum`.  Contraction is off: a fused multiply-add would round once where the separate
// Scale and Sub of the optimizer round twice.
__device__ __forceinline__ float Combine(const GemmF32Args& args, float old, float sum)
{
#pragma clang fp contract(off)
    if (args.sgd != 0)
    {
        const float scaled = sum * args.sgdScale;
        const float step = scaled * args.sgdRate;
        return old - step;
    }
    return old + sum;
}

// Stores acc combined with the old values (or bias terms) `old` for the TM x TN blocks of 32 x 32 one
// wavefront owns, register quad q of block (i, j) at old[(i * TN + j) * 4 + q].
template <int TM, int TN>
__device__ __forceinline__ void FinishTile(const floatx16 (&acc)[TM][TN], float4 (&old)[TM * TN * 4],
                                           float* __restrict__ out, uint32_t rowBase,
                                           uint32_t colBase, uint32_t M, uint32_t N, uint32_t l32,
                                           uint32_t khalf, const GemmF32Args& args)
{
    const bool relu = args.relu != 0;
    const bool inside = rowBase + TM * 32 <= M && colBase + TN * 32 <= N;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
            {
                const uint32_t r = rowBase + i * 32 + l32, c = colBase + j * 32 + 8 * q + 4 * khalf;
                float4 v = old[(i * TN + j) * 4 + q];
                if (!inside && (r >= M || c >= N))
                    continue;
                v.x = Combine(args, v.x, acc[i][j][4 * q + 0]);
                v.y = Combine(args, v.y, acc[i][j][4 * q + 1]);
                v.z = Combine(args, v.z, acc[i][j][4 * q + 2]);
                v.w = Combine(args, v.w, acc[i][j][4 * q + 3]);
                if (relu)
                {
                    v.x = v.x > 0 ? v.x : 0;
                    v.y = v.y > 0 ? v.y : 0;
                    v.z = v.z > 0 ? v.z : 0;
                    v.w = v.w > 0 ? v.w : 0;
                }
                float* p = out + static_cast<size_t>(r) * args.ldc + c;
                if (inside || c + 4 <= N)
                    *reinterpret_cast<floatx4a4*>(p) = floatx4{ v.x, v.y, v.z, v.w };
                else
                {
                    p[0] = v.x;
                    if (c + 1 < N) p[1] = v.y;
                    if (c + 2 < N) p[2] = v.z;
                }
            }
}

// out (+)= acc for the TM x TN blocks of 32 x 32 one wavefront owns; rowBase / colBase are
// the wavefront's first row and column.  Four consecutive columns that all exist are accessed
// 16 bytes at a time, whatever the alignment of the row.
template <int TM, int TN>
__device__ __forceinline__ void StoreTile(const floatx16 (&acc)[TM][TN], float* __restrict__ out,
                                          uint32_t rowBase, uint32_t colBase, uint32_t M,
                                          uint32_t N, uint32_t l32, uint32_t khalf,
                                          const GemmF32Args& args)
{
    const bool accumulate = args.overwrite == 0;
    const float* __restrict__ bias = args.bias;
    // ---- out += acc ---------------------------------------------------------
    // With the operands swapped, register v of lane l holds row l%32 and column
    // 8*(v/4) + 4*(l/32) + v%4 of its 32x32 block: registers 4q..4q+3 are 4
    // consecutive columns.  The old values of the whole wavefront block are requested
    // in one batch, then added and stored.  At the matrix edge the requests stay free of branches
    // too: behind a branch per quad each request was waited for before the next.  Places past the
    // edge read the last row, and the last 4 columns, that exist; a quad that the edge cuts takes
    // its values from those 4 columns (four single floats per quad instead: 1000 x 1000 x 64
    // 5.77 us, this 5.5).
    constexpr int kQuads = TM * TN * 4;
    float4 old[kQuads];
    auto each = [&](auto&& f) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    f(i, j, q, rowBase + i * 32 + l32, colBase + j * 32 + 8 * q + 4 * khalf,
                      old[(i * TN + j) * 4 + q]);
    };
    const bool inside = rowBase + TM * 32 <= M && colBase + TN * 32 <= N;
    if (bias != nullptr)
        // what the K = 1 product ones x bias leaves in a zero-filled out
        each([&](int, int, int, uint32_t, uint32_t c, float4& v) {
            v = make_float4(0.f + bias[min(c, N - 1)], 0.f + bias[min(c + 1, N - 1)],
                            0.f + bias[min(c + 2, N - 1)], 0.f + bias[min(c + 3, N - 1)]);
        });
    else if (!accumulate)
        each([&](int, int, int, uint32_t, uint32_t, float4& v) {
            v = make_float4(0.f, 0.f, 0.f, 0.f);
        });
    else if (inside)
        each([&](int, int, int, uint32_t r, uint32_t c, float4& v) {
            const floatx4 w =
                *reinterpret_cast<const floatx4a4*>(out + static_cast<size_t>(r) * args.ldc + c);
            v = make_float4(w[0], w[1], w[2], w[3]);
        });
    else
    {
        auto rowOf = [&](uint32_t r) {
            return out + static_cast<size_t>(min(r, M - 1)) * args.ldc;
        };
        if (colBase + TN * 32 <= N || N % 4 == 0)  // no quad is cut
            each([&](int, int, int, uint32_t r, uint32_t c, float4& v) {
                const floatx4 w = *reinterpret_cast<const floatx4a4*>(rowOf(r) + min(c, N - 4));
                v = make_float4(w[0], w[1], w[2], w[3]);
            });
        else if (N >= 4)
            each([&](int, int, int, uint32_t r, uint32_t c, float4& v) {
                const uint32_t from = min(c, N - 4), cut = c - from;
                const floatx4 w = *reinterpret_cast<const floatx4a4*>(rowOf(r) + from);
                v.x = cut == 0 ? w[0] : cut == 1 ? w[1] : cut == 2 ? w[2] : w[3];
                v.y = cut == 0 ? w[1] : cut == 1 ? w[2] : w[3];
                v.z = cut == 0 ? w[2] : w[3];
                v.w = w[3];
            });
        else
            each([&](int, int, int, uint32_t r, uint32_t c, float4& v) {
                const float* row = rowOf(r);
                v = make_float4(row[min(c, N - 1)], row[min(c + 1, N - 1)],
                                row[min(c + 2, N - 1)], 0.f);
            });
    }
    FinishTile<TM, TN>(acc, old, out, rowBase, colBase, M, N, l32, khalf, args);
}

// The kernel that takes its operands apart into fp16 planes (sph_gemm_f32_split.hip).  Whether it is the
// faster one for this product, of which the others cost `otherCost`: 107 is what a 64 x 64 tile takes
// on the fp32 matrix cores.
bool SplitsF32(const GemmF32Args& args, uint32_t units, uint64_t otherCost, bool transA, bool transB);
int LaunchGemmF32Split(GemmF32Args args, uint32_t units, bool transA, bool transB,
                       hipStream_t stream);
}  // namespace sph

#endif
