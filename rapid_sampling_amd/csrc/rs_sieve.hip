// Instantiations and launchers of the sieve path.
#include "rs_sieve.h"

namespace rs {

// The finishing workgroup by the units of 64 tokens that the row's slices may set aside, 16 to a wave at most.  (1024 threads with top_k beyond 256, as
// launch_finish has it, were no faster: 128 x 262144 top_k 300 38.3 us a call with them, 34.7 with 256; between 65 and 128 units 128 x 1048576 top_k 1024 takes
// 102.7 us with 1024 threads, 100.5 with 512, 16 x 1048576 top_k 50 23.0 / 22.8.)
static void launch_sieve_finish(uint32_t B, hipStream_t st, const Params &p, const SieveView &v)
{
    const uint32_t n = v.G * v.units;
#define RS_FIN(NTv, PREv) hipLaunchKernelGGL((sieve_finish_kernel<NTv, PREv>), dim3(B), dim3(sieve_finish_threads<NTv>()), 0, st, p, v)
    if (n > 128u) RS_FIN(1024, 16);
    else if (n > 64u) RS_FIN(512, 16);
    else if (n <= 16u) RS_FIN(256, 4);
    else if (n <= 32u) RS_FIN(256, 8);
    else RS_FIN(256, 16);
#undef RS_FIN
}

hipError_t launch_sieve(int R, int32_t dtype, uint32_t B, hipStream_t st, const Params &p, const SieveView &v)
{
    const dim3 grid(B * v.G);
    if (v.G > 128u || v.G * v.units > 256u) return hipErrorInvalidValue;               // what the finishing workgroup asks for
#define RS_SIEVE(Rv, FINEv) do {                                                                                                                \
        if (dtype == RS_DTYPE_F32) hipLaunchKernelGGL((sieve_kernel<Rv, RS_DTYPE_F32, FINEv>), grid, dim3(kThreads), 0, st, p, v);                 \
        else if (dtype == RS_DTYPE_BF16) hipLaunchKernelGGL((sieve_kernel<Rv, RS_DTYPE_BF16, FINEv>), grid, dim3(kThreads), 0, st, p, v);          \
        else hipLaunchKernelGGL((sieve_kernel<Rv, RS_DTYPE_F16, FINEv>), grid, dim3(kThreads), 0, st, p, v); } while (0)
    if (v.fine) { if (R == 16) RS_SIEVE(16, true); else if (R == 8) RS_SIEVE(8, true); else RS_SIEVE(4, true); }
    else { if (R == 16) RS_SIEVE(16, false); else if (R == 8) RS_SIEVE(8, false); else RS_SIEVE(4, false); }
#undef RS_SIEVE
    launch_sieve_finish(B, st, p, v);
    return hipGetLastError();
}

hipError_t launch_sieve_pen(int R, int32_t dtype, uint32_t B, hipStream_t st, const Params &p, const SieveView &v)
{
    const dim3 grid(B * v.G);
    if (v.G > 128u || v.G * v.units > 256u || (R != 4 && R != 8) || v.note_cap != sieve_pen_cap(R) || v.fixers == 0u || (v.G + v.fixers - 1u) / v.fixers > 64u) return hipErrorInvalidValue;
#define RS_SIEVE(Rv, FINEv) do {                                                                                                                     \
        if (dtype == RS_DTYPE_F32) hipLaunchKernelGGL((sieve_pen_kernel<Rv, RS_DTYPE_F32, FINEv>), grid, dim3(kThreads), 0, st, p, v);                  \
        else if (dtype == RS_DTYPE_BF16) hipLaunchKernelGGL((sieve_pen_kernel<Rv, RS_DTYPE_BF16, FINEv>), grid, dim3(kThreads), 0, st, p, v);           \
        else hipLaunchKernelGGL((sieve_pen_kernel<Rv, RS_DTYPE_F16, FINEv>), grid, dim3(kThreads), 0, st, p, v); } while (0)
    if (v.fine) { if (R == 8) RS_SIEVE(8, true); else RS_SIEVE(4, true); }
    else { if (R == 8) RS_SIEVE(8, false); else RS_SIEVE(4, false); }
#undef RS_SIEVE
    launch_sieve_finish(B, st, p, v);
    if (R == 8) hipLaunchKernelGGL((sieve_pen_fix_kernel<8>), dim3(B * v.fixers), dim3(kThreads), 0, st, p, v);
    else hipLaunchKernelGGL((sieve_pen_fix_kernel<4>), dim3(B * v.fixers), dim3(kThreads), 0, st, p, v);
    return hipGetLastError();
}

// What the error bounds of the sieve path's sums rest on, for every float: by how much, in units of 2^-24, the hardware's 2^x is larger than
// e of x, at |x| < 125 (below < 0), or the hardware's 2^(x - M) than e of x for the frame `below` octaves above x, |M| <= 100 (further out x - M is exact,
// and e of it is asked).  out: the least and the largest, in units of 2^-20 of those (both to be set before).
__global__ void __launch_bounds__(kThreads) exp_error_kernel(const int below, long long *out)
{
    const Frame fr(0);
    double least = 1e9, most = -1e9;
    for (uint32_t i = blockIdx.x * kThreads + threadIdx.x; i < 0x42FA0000u; i += gridDim.x * kThreads)
#pragma unroll
        for (uint32_t sign = 0; sign < 2u; ++sign) {
            const float x = __uint_as_float(i | sign << 31), M = below < 0 ? 0.0f : __builtin_floorf(x) + (float)below;
            if (__builtin_fabsf(M) > 100.0f) continue;
            const double e = (double)fr.scaled(x), h = __builtin_ldexp((double)__builtin_amdgcn_exp2f(below < 0 ? x : x - M), (int)M);
            const double off = (h - e) * 0x1p24 / e;
            least = fmin(least, off); most = fmax(most, off);
        }
    atomicMin(&out[0], (long long)floor(least * 0x1p20));
    atomicMax(&out[1], (long long)ceil(most * 0x1p20));
}

hipError_t launch_exp_error(int below, hipStream_t st, long long *out)
{
    hipLaunchKernelGGL(exp_error_kernel, dim3(4096), dim3(kThreads), 0, st, below, out);
    return hipGetLastError();
}

}  // namespace rs
