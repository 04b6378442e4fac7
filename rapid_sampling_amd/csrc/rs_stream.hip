// Instantiations and launchers of the streaming kernels.
#include "rs_stream.h"

namespace rs {

constexpr int kStreamNT = 256;

// The finishing workgroup's size.  Lists of hundreds of tokens (a bounding top_k above 256) out of 32 slices and more: 1024
// threads (128 rows of 1M with top_k 1024: 10.8 us where 256 threads took 13.7; 32 rows of 131072 with top_k 1000, the
// call: 23.0 -> 19.9) while every row has a compute unit to itself (1024 rows of 8192 with top_k 1000: 77 us a call with 1024
// threads, 48 with 256).  Else 256 threads, the scans then stay inside a wave, asking ahead for the first 64 tokens of
// 4, 8 or 16 slices per wave, which is 16 instructions per slice whether the row has it or not (64 rows of 19
// slices: 7.3 us with 16, 6.5 with 8).
static void launch_finish(uint32_t B, size_t lds_bytes, hipStream_t st, const Params &p, const StreamView &v)
{
    if (B <= 256u && v.G >= 32u && p.top_k > 256 && !p.attempt) hipLaunchKernelGGL((finish_kernel<1024, 8>), dim3(B), dim3(finish_threads<1024>()), lds_bytes, st, p, v);
    else if (v.G <= 16u) hipLaunchKernelGGL((finish_kernel<kThreads, 4>), dim3(B), dim3(finish_threads<kThreads>()), lds_bytes, st, p, v);
    else if (v.G <= 32u) hipLaunchKernelGGL((finish_kernel<kThreads, 8>), dim3(B), dim3(finish_threads<kThreads>()), lds_bytes, st, p, v);
    else hipLaunchKernelGGL((finish_kernel<kThreads, 16>), dim3(B), dim3(finish_threads<kThreads>()), lds_bytes, st, p, v);
}

hipError_t launch_stream(int slice_r, int32_t dtype, bool keep, uint32_t B, size_t finish_lds_bytes, hipStream_t st, const Params &p,
                         const StreamView &v)
{
    const dim3 sgrid(B * v.G);
    if (keep && v.G > 2u * kWave) return hipErrorInvalidValue;             // keep_finish_kernel holds two slices per lane
    // keep: the call keeps every live token; what its pass leaves at the head of each slice's stash are masses, and its finish
    // needs no list.
    // NTv threads with Rv groups of four tokens each: a slice of 4 Rv NTv tokens
#ifndef RS_LONG_NT
#define RS_LONG_NT 256
#endif
#define RS_STREAM(Rv, NTv, Lv, KEEPv, PADv) do {                                                                                         \
        if (dtype == RS_DTYPE_F32) hipLaunchKernelGGL((stream_kernel<Rv, NTv, RS_DTYPE_F32, KEEPv, PADv>), sgrid, dim3(NTv), 0, st, p, v);       \
        else if (dtype == RS_DTYPE_BF16) hipLaunchKernelGGL((stream_kernel<Rv, NTv, RS_DTYPE_BF16, KEEPv, PADv>), sgrid, dim3(NTv), 0, st, p, v); \
        else hipLaunchKernelGGL((stream_kernel<Rv, NTv, RS_DTYPE_F16, KEEPv, PADv>), sgrid, dim3(NTv), 0, st, p, v);                             \
        if (KEEPv) hipLaunchKernelGGL((keep_finish_kernel<Lv>), dim3(B), dim3(kKeepT + kWave), 0, st, p, v);                              \
        else launch_finish(B, finish_lds_bytes, st, p, v); } while (0)
    if (slice_r == 4) {
        if (keep) RS_STREAM(4, 256, 12, true, false);
        else if (B * v.G > 256u) RS_STREAM(4, 256, 12, false, true);     // (more workgroups than compute units: see slice_count_and_stash)
        else RS_STREAM(4, 256, 12, false, false);
    }
    else if (slice_r == 8) { if (keep) RS_STREAM(8, 256, 13, true, false); else RS_STREAM(8, 256, 13, false, false); }
    else if (keep) RS_STREAM((kStreamLongR * 256 / RS_LONG_NT), RS_LONG_NT, kStreamLongLog2, true, false);
    else {
        // (a quarter of the slots past the ends of their rows: see slice_count_and_stash)
        const uint32_t slots = v.G << kStreamLongLog2;
        if (slots - (uint32_t)p.V >= slots >> 2) RS_STREAM((kStreamLongR * 256 / RS_LONG_NT), RS_LONG_NT, kStreamLongLog2, false, true);
        else RS_STREAM((kStreamLongR * 256 / RS_LONG_NT), RS_LONG_NT, kStreamLongLog2, false, false);
    }
#undef RS_STREAM
    return hipGetLastError();
}

hipError_t launch_stream_pen(int slice_r, uint32_t B, size_t finish_lds_bytes, hipStream_t st, const Params &p, const StreamView &v)
{
    if (slice_r == 8) hipLaunchKernelGGL((stream_pen_kernel<8>), dim3(B * v.G), dim3(kThreads), 0, st, p, v);
    else hipLaunchKernelGGL((stream_pen_kernel<kStreamLongR>), dim3(B * v.G), dim3(kThreads), 0, st, p, v);
    launch_finish(B, finish_lds_bytes, st, p, v);
    return hipGetLastError();
}

hipError_t launch_penalty_fix(int slice_r, hipStream_t st, const Params &p, const StreamView &v)
{
    if (slice_r == 8) hipLaunchKernelGGL((penalty_fix_kernel<8>), dim3((uint32_t)p.B * v.G), dim3(kThreads), 0, st, p, v);
    else hipLaunchKernelGGL((penalty_fix_kernel<kStreamLongR>), dim3((uint32_t)p.B * v.G), dim3(kThreads), 0, st, p, v);
    return hipGetLastError();
}

hipError_t launch_fused(int slice_r, bool pen, uint32_t B, hipStream_t st, const Params &p, const StreamView &v)
{
    const dim3 grid(B * v.G), block(kThreads);
    if (v.list_cap > 2048u) return hipErrorInvalidValue;      // the list lives in static LDS
    // (slices asked for ahead: launch_finish)
#define RS_FUSED_PRE(Rv, PREv) do { if (pen) hipLaunchKernelGGL((fused_kernel<Rv, true, PREv>), grid, block, 0, st, p, v);          \
                                    else hipLaunchKernelGGL((fused_kernel<Rv, false, PREv>), grid, block, 0, st, p, v); } while (0)
#define RS_FUSED(Rv) do { if (v.G <= 16u) RS_FUSED_PRE(Rv, 4); else if (v.G <= 32u) RS_FUSED_PRE(Rv, 8); else RS_FUSED_PRE(Rv, 16); } while (0)
    switch (slice_r) {
    case 4:  RS_FUSED(4); break;
    case 8:  RS_FUSED(8); break;
    default: RS_FUSED(16); break;
    }
#undef RS_FUSED
#undef RS_FUSED_PRE
    return hipGetLastError();
}

}  // namespace rs
