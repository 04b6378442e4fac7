// The sieve path's records in the workspace, and its launcher.
#pragma once

#include "rs_common.h"

namespace rs {

struct SieveHdr {                                        // 16 bytes
    uint32_t mkey;           // fkey(max x of the slice)
    uint32_t n;              // tokens set aside; kSieveTie: none, and all tokens of the slice equal its maximum
    uint32_t cut;            // every token of the slice with fkey(x) > cut is set aside
    uint32_t mass;           // float: the sum of 2^(x - floor(max x))
};
constexpr uint32_t kSieveTie = 1u << 31, kSieveOdd = 1u << 30;     // kSieveOdd, with any n: a wave's sum was worked out in a frame

struct SieveView {
    SieveHdr *hdr;           // [B][G]
    uint64_t *stash;         // [B][G][64 * units]   bits of x << 32 | index, in no order
    uint32_t  G;             // slices per row
    uint32_t  units;         // a slice sets aside at most 64 tokens (1) or 128 (2)
    uint32_t  reach;         // pairs of threads, of a slice's 128, whose largest token is set aside
};

// R: groups of four tokens of a lane, 4, 8 or 16: slices of 256 R tokens
hipError_t launch_sieve(int R, int32_t dtype, uint32_t B, hipStream_t st, const Params &p, const SieveView &v);

}  // namespace rs
