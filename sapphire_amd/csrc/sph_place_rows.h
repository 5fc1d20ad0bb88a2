// Row offsets and the move of staged rows in one launch.
//
// A pass that cannot know where its rows go (the counts of all rows above decide that) leaves
// every row's entries in a staging slot and its count in an array.  A scan of the counts followed
// by a kernel that moves the rows is two to four dependent launches of 4 to 7 us each, nearly all
// of it launch latency and a single workgroup's serial rounds.  Here every workgroup adds up the
// counts of all rows above its own by itself -- up to kPlaceMaxRows counts of 4 bytes, out of the
// L2 -- scans its own rows, writes their offsets and moves them.  The repeated reading grows
// with the square of the rows (65536 rows: 64 MiB over all workgroups), so longer arrays are
// scanned by launches of their own.  The counts must not be the array of offsets itself:
// other workgroups still read them.
#ifndef SPH_PLACE_ROWS_H
#define SPH_PLACE_ROWS_H

#include "sph_internal.h"

#include <algorithm>

namespace sph
{
constexpr uint32_t kPlaceThreads = 1024;
constexpr uint32_t kPlaceWaves = kPlaceThreads / 64;
constexpr uint32_t kPlaceMaxRows = 1u << 17;

// Rows per workgroup: at most two workgroups per compute unit (all resident), a multiple of 4 so
// that the counts above a workgroup's rows are whole 16-byte quads, at most one row per thread.
inline uint32_t PlaceRowsPerGroup(uint32_t M)
{
    const uint32_t groups = static_cast<uint32_t>(ComputeUnits()) * 2;
    const uint32_t rows = std::max<uint32_t>(kPlaceWaves, (M + groups - 1) / groups);
    return std::min<uint32_t>((rows + 3) / 4 * 4, kPlaceThreads);
}

// LDS of one workgroup
struct PlaceScratch
{
    uint32_t waveAbove[kPlaceWaves], waveOwn[kPlaceWaves];
    uint32_t offset[kPlaceThreads + 1];  // of the workgroup's own rows, and the end of the last
};

// Writes ROW for the workgroup's rows (and ROW[M] in the last workgroup) and leaves them in
// lds.offset.  All threads of the workgroup take part; counts is 16-byte aligned.
__device__ __forceinline__ void PlaceOffsets(uint32_t* __restrict__ ROW,
                                             const uint32_t* __restrict__ counts, uint32_t M,
                                             uint32_t rowsPerGroup, PlaceScratch& lds)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t first = blockIdx.x * rowsPerGroup;
    const uint4* quads = reinterpret_cast<const uint4*>(counts);
    uint32_t above = 0;
#pragma unroll 4
    for (uint32_t q = threadIdx.x; q < first / 4; q += kPlaceThreads)
    {
        const uint4 c = quads[q];
        above += c.x + c.y + c.z + c.w;
    }
    const bool own = threadIdx.x < rowsPerGroup && first + threadIdx.x < M;
    const uint32_t count = own ? counts[first + threadIdx.x] : 0u;
    uint32_t inclusive = count;
#pragma unroll
    for (uint32_t d = 1; d < 64; d *= 2)
    {
        above += __shfl_xor(above, d, 64);
        const uint32_t left = __shfl_up(inclusive, d, 64);
        if (lane >= d)
            inclusive += left;
    }
    if (lane == 63)
    {
        lds.waveAbove[wave] = above;
        lds.waveOwn[wave] = inclusive;
    }
    __syncthreads();
    uint32_t start = 0;
#pragma unroll
    for (uint32_t w = 0; w < kPlaceWaves; ++w)
        start += lds.waveAbove[w] + (w < wave ? lds.waveOwn[w] : 0u);
    const uint32_t end = start + inclusive;
    if (own)
    {
        ROW[first + threadIdx.x] = end - count;
        lds.offset[threadIdx.x] = end - count;
        if (threadIdx.x == rowsPerGroup - 1 || first + threadIdx.x == M - 1)
            lds.offset[threadIdx.x + 1] = end;
        if (first + threadIdx.x == M - 1)
            ROW[M] = end;
    }
    __syncthreads();
}

// One wavefront moves rows of up to `slot` staged entries: rows r0, r0 + kPlaceWaves, ... of its
// workgroup, four at a time so that their loads are in flight together.  `overfull(row, begin,
// end)` gets the rows that did not fit their slot.  Nothing is stored at or past `capacity`.
template <typename Overfull>
__device__ __forceinline__ void MoveStagedRows(float* __restrict__ V, uint32_t* __restrict__ COL,
                                               const float* __restrict__ stageV,
                                               const uint32_t* __restrict__ stageCol, uint32_t M,
                                               uint32_t rowsPerGroup, uint32_t slot,
                                               uint32_t capacity, const PlaceScratch& lds,
                                               Overfull&& overfull)
{
    constexpr uint32_t kTogether = 4;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t first = blockIdx.x * rowsPerGroup;
    const uint32_t rows = first < M ? min(rowsPerGroup, M - first) : 0u;
    for (uint32_t r0 = threadIdx.x >> 6; r0 < rows; r0 += kPlaceWaves * kTogether)
    {
        float v[kTogether];
        uint32_t c[kTogether];
#pragma unroll
        for (uint32_t u = 0; u < kTogether; ++u)
        {
            const uint32_t r = r0 + u * kPlaceWaves;
            v[u] = 0.0f;
            c[u] = 0;
            const uint32_t n = r < rows ? lds.offset[r + 1] - lds.offset[r] : 0u;
            if (n <= slot && lane < n)
            {
                const size_t from = static_cast<size_t>(first + r) * slot + lane;
                v[u] = stageV[from];
                c[u] = stageCol[from];
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < kTogether; ++u)
        {
            const uint32_t r = r0 + u * kPlaceWaves;
            if (r >= rows)
                break;
            const uint32_t to = lds.offset[r];
            const uint32_t n = lds.offset[r + 1] - to;
            if (n > slot)
            {
                overfull(first + r, to, to + n);
                continue;
            }
            if (lane < n && to + lane < capacity)
            {
                V[to + lane] = v[u];
                COL[to + lane] = c[u];
            }
            const size_t from = static_cast<size_t>(first + r) * slot;
            for (uint32_t i = lane + 64; i < n; i += 64)
                if (to + i < capacity)
                {
                    V[to + i] = stageV[from + i];
                    COL[to + i] = stageCol[from + i];
                }
        }
    }
}
}  // namespace sph

#endif
