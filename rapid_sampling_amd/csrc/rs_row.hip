// Instantiations and the launcher of the row kernel.
#include "rs_row.h"

namespace rs {

constexpr uint32_t kCUs = 256u;        // of an MI355X

template <int NT, int R>
static void launch_row_r(int32_t dtype, uint32_t B, hipStream_t st, const Params &p)
{
    if (dtype == RS_DTYPE_F32) hipLaunchKernelGGL((row_kernel<RS_DTYPE_F32, NT, R>), dim3(B), dim3(NT), 0, st, p);
    else if (dtype == RS_DTYPE_BF16) hipLaunchKernelGGL((row_kernel<RS_DTYPE_BF16, NT, R>), dim3(B), dim3(NT), 0, st, p);
    else hipLaunchKernelGGL((row_kernel<RS_DTYPE_F16, NT, R>), dim3(B), dim3(NT), 0, st, p);
}

// Groups of four tokens per thread: the fewest of 2, 4, 8, 13 and 16 that hold the row (13: rows of 50304 tokens).
// More rows than compute units: rows of up to 32768 tokens with half the threads and twice the groups each, two
// rows to a compute unit (registers and LDS hold two such workgroups, but only one of 1024 threads), so that one
// row's scans, barriers and one-thread steps run beside the other's counting: 512 rows of 32768 float16 39.6 -> 31.3
// us a call.  (Two workgroups of 1024 threads in 64 registers each spill: 44.3.)  Up to 256 rows every row has a compute
// unit to itself, and 1024 threads are the faster there.
hipError_t launch_row(int32_t dtype, uint32_t B, hipStream_t st, const Params &p)
{
    if (p.V <= 0 || p.V > kRowMaxV || (p.V & 3)) return hipErrorInvalidValue;
    const uint32_t need = (((uint32_t)p.V >> 2) + (uint32_t)kRowW - 1u) / (uint32_t)kRowW;   // groups per wave of sixteen
    if (B > kCUs && need <= 8u * kWave) {
        const uint32_t need8 = (((uint32_t)p.V >> 2) + 7u) / 8u;                             // ... of eight
        if (need8 <= 4u * kWave) launch_row_r<512, 4>(dtype, B, st, p);
        else if (need8 <= 8u * kWave) launch_row_r<512, 8>(dtype, B, st, p);
        else if (need8 <= 12u * kWave) launch_row_r<512, 12>(dtype, B, st, p);
        else launch_row_r<512, 16>(dtype, B, st, p);
    } else if (need <= 2u * kWave) launch_row_r<1024, 2>(dtype, B, st, p);
    else if (need <= 4u * kWave) launch_row_r<1024, 4>(dtype, B, st, p);
    else if (need <= 8u * kWave) launch_row_r<1024, 8>(dtype, B, st, p);
    else if (need <= 13u * kWave) launch_row_r<1024, 13>(dtype, B, st, p);
    else launch_row_r<1024, 16>(dtype, B, st, p);
    return hipGetLastError();
}

}  // namespace rs
