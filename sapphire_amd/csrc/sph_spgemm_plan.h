// Arithmetic of the CSR x CSR launches that the kernels and the host share, in one place so that
// the CPU tests exercise what runs on the device.
#ifndef SPH_SPGEMM_PLAN_H
#define SPH_SPGEMM_PLAN_H

#include <cstddef>
#include <cstdint>

#if defined(__HIPCC__)
#define SPH_PLAN_HOST_DEVICE __host__ __device__
#else
#define SPH_PLAN_HOST_DEVICE
#endif

namespace sph
{
// Turns of rowsPerTurn (at least 1) consecutive rows that M rows make, the last one possibly
// short.  No rows make no turn, and nothing wraps for any M.
SPH_PLAN_HOST_DEVICE inline uint32_t SpgemmTurns(uint32_t M, uint32_t rowsPerTurn)
{
    return M / rowsPerTurn + (M % rowsPerTurn != 0 ? 1u : 0u);
}

// Staging slots, in entries per row, that the one-call product tries in turn until `take(slot)`
// finds memory for them: three times the mean row that the capacity allows plus 64, then twice the
// mean.  All M slots together stay below 2^31 entries.  Returns the slot taken, 0 for none: the
// products are then counted first and computed a second time to be stored.
// Twice the mean is too little for rows whose lengths vary like those of a random graph: of
// 65536 rows with 64 products on average one or two did not fit and were done again.
template <typename Take>
uint32_t TakeStagingSlot(uint32_t M, uint32_t N, uint32_t capacity, Take&& take)
{
    if (M == 0 || N == 0 || capacity == 0)
        return 0;
    const uint64_t mean = capacity / M;
    for (uint64_t times = 3; times >= 2; --times)
    {
        const uint64_t slot = times * mean + 64;
        if (slot * M < (1ull << 31) && take(static_cast<uint32_t>(slot)))
            return static_cast<uint32_t>(slot);
    }
    return 0;
}

// Bytes of a staging block that is to stay for the next call, which may need a little more: a quarter
// on top, up to `most`, where `take(bytes)` finds memory for that, else just `bytes` (<= most).  Returns
// what was taken, 0 for nothing.
template <typename Take>
std::size_t TakeWithRoom(std::size_t bytes, std::size_t most, Take&& take)
{
    const std::size_t more = bytes + bytes / 4 < most ? bytes + bytes / 4 : most;
    if (take(more))
        return more;
    return more != bytes && take(bytes) ? bytes : 0;
}
}  // namespace sph

#endif
