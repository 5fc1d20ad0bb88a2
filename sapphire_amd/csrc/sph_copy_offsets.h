// Where the tiled GEMM kernels copy the chunks of an operand from, when its rows are no whole number of
// chunks or steps.  One definition for the kernels and for the host, so that the CPU tests
// see that no copy reaches past an operand: what it would bring feeds no output and shows in none.
//
// Operand stored k-major: a row's last chunk reaches into the next row, whose values only feed outputs that are not
// stored.  In the last row of the matrix there is none; the chunk begins earlier there, so that it
// ends with the row.  Chunks past a row's end copy its last whole chunk.
#ifndef SPH_COPY_OFFSETS_H
#define SPH_COPY_OFFSETS_H

#include <cstdint>

#if defined(__HIPCC__)
#define SPH_COPY_INLINE __host__ __device__ inline __attribute__((always_inline))
#else
#define SPH_COPY_INLINE inline
#endif

namespace sph
{
struct KMajorPlace
{
    uint32_t k, column;
};

// fp32, chunks of 4: where the chunk for column x of row k of a slab is copied from.  `valid` rows of
// the slab exist (those past them copy the first one); `ending`: its last one is the matrix's.
// limit >= 4 columns.
SPH_COPY_INLINE KMajorPlace QuadPlace(uint32_t k, uint32_t x, uint32_t limit, uint32_t valid,
                                      bool ending)
{
    if (k >= valid)
        k = 0;
    const uint32_t last = limit - 4;
    const bool clamp = x >= limit || (ending && k + 1 == valid);
    return { k, clamp && x > last ? last : x };
}

// fp32, an operand stored with K contiguous: chunk c of a row of a slab that has `valid` values of k ends
// with this one.  Chunks that reach past `valid`, and those that begin past it, are the row's last four
// values, whatever `valid` is (K >= 4): up to three of them lie before the slab.
SPH_COPY_INLINE uint32_t RowChunkEnd(uint32_t c, uint32_t valid)
{
    const uint32_t end = c * 4 + 4;
    return end < valid ? end : valid;
}

// fp32, few rows of an operand stored k-major: `floats` values that lie one behind the other, in pieces of
// 4.  Of `slots` pieces that are asked for at once those past the end are the last whole one again;
// where there is none, no piece is asked for.
SPH_COPY_INLINE uint32_t PiecesAsked(uint32_t floats, uint32_t slots)
{
    return floats < 4 ? 0 : slots;
}

SPH_COPY_INLINE uint32_t PieceBegin(uint32_t piece, uint32_t floats)
{
    return piece * 4 < floats - 4 ? piece * 4 : floats - 4;
}

// fp16, chunks of 8 (x a multiple of 8, limit >= 8): the first column a chunk is copied from, in every
// row but the last of the matrix
SPH_COPY_INLINE uint32_t ChunkColumn(uint32_t x, uint32_t limit)
{
    return x < limit ? x : limit - 8;
}

// ... and the bytes by which it has to begin earlier there
SPH_COPY_INLINE uint32_t LastChunkBack(uint32_t x, uint32_t limit)
{
    return x < limit && x + 8 > limit ? (x + 8 - limit) * 2 : 0u;
}
}  // namespace sph

#endif
