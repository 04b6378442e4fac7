// The sieve path's records in the workspace, and its launcher.
#pragma once

#include "rs_common.h"

namespace rs {

struct SieveHdr {                                        // 16 bytes
    uint32_t mkey;           // fkey(max x of the slice)
    uint32_t n;              // tokens set aside; kSieveTie: none, and all tokens of the slice equal its maximum
    uint32_t cut;            // every token of the slice with fkey(x) > cut is set aside
    uint32_t mass;           // float: the sum of 2^(x - floor(max x)); kSieveOdd in the place of its sign: a wave's was worked out in a frame, one that matters
};
constexpr uint32_t kSieveTie = 1u << 31, kSieveOdd = 1u << 31;

struct SieveFine {                                       // 16 bytes
    double   mass;           // the sum of the slice's e, in its frame
    uint32_t low;            // fkey(min x of the slice)
    uint32_t pad;
};

struct SieveView {
    SieveHdr *hdr;           // [B][G]
    SieveFine *fine;         // [B][G], or null: the passes' sums are those of the headers
    uint64_t *stash;         // [B][G][64 * units]   bits of x << 32 | index, in no order
    uint32_t  G;             // slices per row
    uint32_t  units;         // a slice sets aside at most 64 tokens (1) or 128 (2)
    uint32_t  reach;         // pairs of threads, of a slice's 128, whose largest token is set aside
    uint32_t  keep;          // tokens that a slice with more than it has room for sets aside at least
    // calls with penalties: the groups of four of which one penalty's bit pattern is not +0.0, as they were
    uint32_t *noted;         // [B][G][4]            how many a wave has noted, or kSievePenLeft
    uint32_t *note_at;       // [B][G][4][note_cap]  which groups of the row
    float4   *note_old;      // [B][G][4][note_cap]  their penalties
    uint32_t  note_cap;      // sieve_pen_cap of the slices' length
    uint32_t  fixers;        // workgroups of the fix-up kernel to a row
};
constexpr uint32_t kSievePenLeft = 0xFFFFFFFFu;          // the wave's penalties are still the old ones: to be rewritten by the fix-up kernel
// Of a wave's 64 R groups, 11 in 64: some 4 % of the tokens by chance, or 17 % side by side; as many as a workspace of rs_workspace_bytes has room
// for in rows of a million tokens.
__host__ __device__ constexpr uint32_t sieve_pen_cap(int R) { return 11u * (uint32_t)R; }

// R: groups of four tokens of a thread, 4, 8 or 16: slices of 1024 R tokens; with penalties 4 or 8
hipError_t launch_sieve_pen(int R, int32_t dtype, uint32_t B, hipStream_t st, const Params &p, const SieveView &v);
hipError_t launch_sieve(int R, int32_t dtype, uint32_t B, hipStream_t st, const Params &p, const SieveView &v);
hipError_t launch_exp_error(int below, hipStream_t st, long long *out);

}  // namespace rs
