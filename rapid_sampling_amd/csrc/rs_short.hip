// Instantiations and the launcher of the short-row kernel.
#include "rs_short.h"

namespace rs {

constexpr uint32_t kCUs = 256u;        // of an MI355X

template <int W, int R>
static void launch_short_r(bool pen, int32_t dtype, uint32_t B, hipStream_t st, const Params &p)
{
    const dim3 grid(B), block(short_threads<W>());
#define RS_SHORT(DTv) do { if (pen) hipLaunchKernelGGL((short_kernel<DTv, true, W, R>), grid, block, 0, st, p);          \
                           else hipLaunchKernelGGL((short_kernel<DTv, false, W, R>), grid, block, 0, st, p); } while (0)
    if (dtype == RS_DTYPE_F32) RS_SHORT(RS_DTYPE_F32);
    else if (dtype == RS_DTYPE_BF16) RS_SHORT(RS_DTYPE_BF16);
    else RS_SHORT(RS_DTYPE_F16);
#undef RS_SHORT
}

// Waves per row and groups of four tokens per thread.  While every row has a compute unit to itself the fewest tokens per
// thread are the fastest, until sixteen waves cost more in barriers than they save (64 rows, top_k 40 / a wide nucleus, 4, 8 and 16
// waves: 4096 tokens 6.0 6.1 5.8 / 9.2 8.1 8.3 us a call, 8192 tokens 7.4 6.7 6.5 / 13.5 10.3 9.8, 16384 - 8.6 8.0 / - 15.2 13.2);
// with more rows than compute units the smaller workgroups are, several of them to a compute unit (1024 rows of 4096:
// 8.7 14.5 12.7 / 14.3 18.8 21.2; 1024 of 8192 with penalties: 31.2 27.8 29.8 / 37.7 31.6 39.8).  Rows of up to 12288 tokens
// have three groups a thread, not four, the last of which would be empty: with penalties 2048 rows of 8196 102 -> 91, 64 13.2 -> 12.0; without
// 64 rows of 8196, top_k 1000 12.3 -> 11.3.
hipError_t launch_short(bool pen, int32_t dtype, uint32_t B, hipStream_t st, const Params &p)
{
    if (p.V <= 0 || p.V > kShortMaxV || (p.V & 3)) return hipErrorInvalidValue;
    if (p.V <= 1024) launch_short_r<4, 1>(pen, dtype, B, st, p);
    else if (B > kCUs && p.V <= 2048) launch_short_r<4, 2>(pen, dtype, B, st, p);
    else if (B > kCUs && p.V <= 4096) launch_short_r<4, 4>(pen, dtype, B, st, p);
    else if (B > kCUs && p.V <= 8192) launch_short_r<8, 4>(pen, dtype, B, st, p);
    else if (p.V <= 2048) launch_short_r<8, 1>(pen, dtype, B, st, p);
    else if (p.V <= 4096) launch_short_r<8, 2>(pen, dtype, B, st, p);
    else if (p.V <= 8192) launch_short_r<16, 2>(pen, dtype, B, st, p);
    else if (p.V <= 12288) launch_short_r<16, 3>(pen, dtype, B, st, p);
    else launch_short_r<16, 4>(pen, dtype, B, st, p);
    return hipGetLastError();
}

}  // namespace rs
