// Arithmetic of the CSR x CSR launches that the kernels and the host share, in one place so that
// the CPU tests exercise what runs on the device.
#ifndef SPH_SPGEMM_PLAN_H
#define SPH_SPGEMM_PLAN_H

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
}  // namespace sph

#endif
