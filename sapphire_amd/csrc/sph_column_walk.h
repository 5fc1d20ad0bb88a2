// How a group of lanes walks the columns of one row in the dense -> CSR count and fill passes.
// One definition for the kernels and for the host, so that the CPU tests exercise the arithmetic
// that runs on the device.
//
// A step hands `step` consecutive columns to the group (4 per lane).  While `ahead` whole steps
// are left they are taken as one batch, whose loads are in flight together; the rest goes step by
// step.  The batches compare against N less one batch: `first + ahead * step <= N` wraps for N
// within a batch of 2^32 and never ends.  The single steps stop at N rounded up to a whole step,
// which 32 bits hold for N up to kMaxColumns.
#ifndef SPH_COLUMN_WALK_H
#define SPH_COLUMN_WALK_H

#include <cstdint>

#if defined(__HIPCC__)
#define SPH_WALK_INLINE __host__ __device__ inline __attribute__((always_inline))
#else
#define SPH_WALK_INLINE inline
#endif

namespace sph
{
// widest row of the walk: a step is at most 256 columns
constexpr uint32_t kMaxColumns = 0xffffff00u;

// batch(first): columns first .. first + ahead * step - 1, all below N.
// single(first): columns first .. first + step - 1, those below N.
template <typename Batch, typename Single>
SPH_WALK_INLINE void WalkColumns(uint32_t N, uint32_t step, uint32_t ahead, Batch&& batch,
                                 Single&& single)
{
    uint32_t first = 0;
    if (N >= ahead * step)
        for (const uint32_t last = N - ahead * step; first <= last; first += ahead * step)
            batch(first);
    for (; first < N; first += step)
        single(first);
}
}  // namespace sph

#endif
