// 96-bit masses (a row's total weight stays below 2^84) and the scan of a histogram by one wave.
#pragma once

#include "rs_common.h"

namespace rs {

// ---- 96-bit masses ------------------------------------------------------------
struct M96 {
    uint64_t lo;
    uint32_t hi;
};
__device__ __forceinline__ M96 m96(u128 v) { return M96{(uint64_t)v, (uint32_t)(v >> 64)}; }
__device__ __forceinline__ u128 wide(M96 a) { return ((u128)a.hi << 64) | a.lo; }
__device__ __forceinline__ M96 operator+(M96 a, M96 b)
{
    M96 r;
    const bool c = __builtin_add_overflow(a.lo, b.lo, &r.lo);
    r.hi = a.hi + b.hi + (c ? 1u : 0u);
    return r;
}
__device__ __forceinline__ M96 operator-(M96 a, M96 b)
{
    M96 r;
    const bool c = __builtin_sub_overflow(a.lo, b.lo, &r.lo);
    r.hi = a.hi - b.hi - (c ? 1u : 0u);
    return r;
}
__device__ __forceinline__ bool operator>=(M96 a, M96 b) { return a.hi > b.hi || (a.hi == b.hi && a.lo >= b.lo); }
__device__ __forceinline__ bool operator<(M96 a, M96 b) { return !(a >= b); }

__device__ __forceinline__ uint32_t lane_of(uint32_t v, uint32_t l) { return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l); }
__device__ __forceinline__ uint64_t lane_of(uint64_t v, uint32_t l) { return ((uint64_t)lane_of((uint32_t)(v >> 32), l) << 32) | lane_of((uint32_t)v, l); }
__device__ __forceinline__ M96 lane_of(M96 v, uint32_t l) { return M96{lane_of(v.lo, l), lane_of(v.hi, l)}; }
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ uint64_t uniform(uint64_t v) { return ((uint64_t)uniform((uint32_t)(v >> 32)) << 32) | uniform((uint32_t)v); }
__device__ __forceinline__ M96 uniform(M96 v) { return M96{uniform(v.lo), uniform(v.hi)}; }

// Mass of a packed bin whose tokens share the exponent ex (87 <= ex <= 127): 44 bits shifted by up to 40.
__device__ __forceinline__ M96 pack_m96(uint64_t w, uint32_t ex)
{
    const uint64_t sum = (w & kPackMask) + ((w >> 43) << 23);
    const uint32_t sh = ex - 87u;
    return M96{sum << sh, (uint32_t)((sum >> 24) >> (40u - sh))};
}

// The same mass as four limbs of 24 bits in 32-bit words: sums of up to 256 of them need no carries, so a scan
// over a wave is four independent chains of fused DPP adds (a 96-bit add costs a carry through the VCC register
// per word, with wait states between).
struct Limbs {
    uint32_t w[4];
};
__device__ __forceinline__ Limbs operator+(Limbs a, Limbs b) { return Limbs{{a.w[0] + b.w[0], a.w[1] + b.w[1], a.w[2] + b.w[2], a.w[3] + b.w[3]}}; }
__device__ __forceinline__ Limbs operator-(Limbs a, Limbs b) { return Limbs{{a.w[0] - b.w[0], a.w[1] - b.w[1], a.w[2] - b.w[2], a.w[3] - b.w[3]}}; }
__device__ __forceinline__ Limbs limbs(M96 m)
{
    const uint32_t x = (uint32_t)m.lo, y = (uint32_t)(m.lo >> 32), z = m.hi;
    return Limbs{{x & 0xFFFFFFu, __builtin_amdgcn_alignbit(y, x, 24u) & 0xFFFFFFu, __builtin_amdgcn_alignbit(z, y, 16u) & 0xFFFFFFu, z >> 8}};
}
__device__ __forceinline__ M96 m96(Limbs l)
{
    const uint32_t w1 = l.w[1] + (l.w[0] >> 24), w2 = l.w[2] + (w1 >> 24), w3 = l.w[3] + (w2 >> 24);
    const uint32_t x = (l.w[0] & 0xFFFFFFu) | w1 << 24, y = (w1 >> 8 & 0xFFFFu) | w2 << 16, z = (w2 >> 16 & 0xFFu) | w3 << 8;
    return M96{((uint64_t)y << 32) | x, z};
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ void dpp_add(Limbs &v)
{
#pragma unroll
    for (int i = 0; i < 4; ++i) v.w[i] += dpp0_u32<CTRL, ROW_MASK>(v.w[i]);
}
__device__ __forceinline__ Limbs wave_inclusive_scan(Limbs v)
{
    dpp_add<0x111, 0xf>(v); dpp_add<0x112, 0xf>(v); dpp_add<0x114, 0xf>(v); dpp_add<0x118, 0xf>(v);
    dpp_add<0x142, 0xa>(v); dpp_add<0x143, 0xc>(v);
    return v;
}
__device__ __forceinline__ Limbs lane_of(Limbs v, uint32_t l) { return Limbs{{lane_of(v.w[0], l), lane_of(v.w[1], l), lane_of(v.w[2], l), lane_of(v.w[3], l)}}; }

// ceil(f * s) for a uniform s < 2^96 and a float 0 < f <= 1 (see ceil_mul), the usual 2^-7 <= f < 1 by one 32-bit multiplication
// per word.
__device__ __forceinline__ M96 ceil_mul(float f, M96 s)
{
    const uint32_t fb = __float_as_uint(f), sh = 150u - (fb >> 23);              // f = m * 2^-sh
    if (sh - 24u < 8u) {
        const uint64_t m = (fb & 0x7FFFFFu) | 0x800000u;
        const uint64_t p0 = m * (uint32_t)s.lo + ((1ull << sh) - 1ull);          // (below 2^56 + 2^31)
        const uint64_t p1 = m * (uint32_t)(s.lo >> 32) + (p0 >> 32), p2 = m * s.hi + (p1 >> 32);
        const uint64_t lo = (p1 << 32) | (uint32_t)p0;
        return M96{(lo >> sh) | (p2 << (64u - sh)), (uint32_t)(p2 >> sh)};
    }
    return m96(ceil_mul(f, wide(s)));
}

// A histogram looked at by one wave, K <= 3 bins per lane, largest e first: counts and masses per bin and
// summed over the lanes before.
template <int K>
struct BinScan {
    uint32_t c[K], before;
    Limbs    m[K], mb, mi;                               // mb: mass of the lanes before; mi: that and this lane's own
    // bin(i): packed word of the lane's i-th bin; ex(i): its exponent
    template <typename BIN, typename EX>
    __device__ __forceinline__ void load(BIN bin, EX ex)
    {
        uint32_t cs = 0;
        Limbs ms{{0u, 0u, 0u, 0u}};
        uint64_t w[K];
#pragma unroll
        for (int i = 0; i < K; ++i) w[i] = bin(i);
#pragma unroll
        for (int i = 0; i < K; ++i) {
            c[i] = pack_count(w[i]);
            m[i] = limbs(pack_m96(w[i], ex(i)));
            cs += c[i]; ms = ms + m[i];
        }
        before = wave_inclusive_scan(cs) - cs;
        mi = wave_inclusive_scan(ms);
        mb = mi - ms;
    }
    __device__ __forceinline__ M96 total() const { return m96(lane_of(mi, 63u)); }
    // The first bin at which (cnt0 + count so far >= top_k) or (mass0 + mass so far >= P): its place in scan
    // order, what lies before it, its count (all wave-uniform); returns false when there is none.
    __device__ __forceinline__ bool search(uint32_t cnt0, M96 mass0, uint32_t top_k, M96 P, uint32_t &place, uint32_t &cnt_above,
                                           uint32_t &cnt_bin, M96 &mass_above) const
    {
        uint32_t run = cnt0 + before;
        Limbs mr = mb + limbs(mass0);
        bool after[K];
#pragma unroll
        for (int i = 0; i < K; ++i) {
            run += c[i]; mr = mr + m[i];
            const M96 q = m96(mr);
            after[i] = run >= top_k || q >= P;
        }
        const uint64_t vote = __builtin_amdgcn_ballot_w64(after[K - 1]);
        if (vote == 0ull) return false;
        const uint32_t l = (uint32_t)__builtin_ctzll(vote);
        // the lane's own bins one after the other, on scalars
        uint32_t i = 0;
        cnt_above = cnt0 + lane_of(before, l); cnt_bin = lane_of(c[0], l);
        Limbs ma = lane_of(mb, l) + limbs(mass0);
#pragma unroll
        for (int k = 0; k + 1 < K; ++k)
            if (!(__builtin_amdgcn_ballot_w64(after[k]) >> l & 1ull)) {
                cnt_above += cnt_bin; cnt_bin = lane_of(c[k + 1], l); ma = ma + lane_of(m[k], l);
                i = (uint32_t)k + 1u;
            }
        place = l * (uint32_t)K + i;
        mass_above = m96(ma);
        return true;
    }
};

}  // namespace rs
