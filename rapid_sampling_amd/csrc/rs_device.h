// Device-side building blocks of the MI355X token sampler: canonical
// element-wise arithmetic, wave64 reductions and scans on the DPP data path,
// Philox.
//
// Arithmetic contract (shared with the CPU oracle used by the tests): every
// floating-point step is a single IEEE fp32 operation (compile with
// -ffp-contract=off; fused multiply-adds are explicit), and everything summed
// across tokens is an integer, so no result depends on how tokens are spread
// over lanes, waves or workgroups.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rs {

constexpr int kWave = 64;

// ---------------------------------------------------------------- scalars --

// NaN -> 0, +-Inf -> +-FLT_MAX            (reference: sampling.cu:131-134)
__device__ __forceinline__ float sf(float x)
{
    float y = (x != x) ? 0.0f : x;
    return fminf(fmaxf(y, -3.402823466e+38f), 3.402823466e+38f);
}

typedef unsigned __int128 u128;

constexpr uint32_t kEMinBits = 0x2B800000u;               // bit pattern of 2^-40, the smallest live e
constexpr uint32_t kDeadBits = 0x2B000000u;               // 2^-41: where the registers keep what lies below

// A token whose e falls below 2^-40 is DEAD: its probability is exactly 0 (the reference's
// exp2f(x - max) underflows to 0 likewise, 149 octaves down, sampling.cu:235), it takes no part
// in the selection and can never be returned -- a logit masked with -inf must not come back
// however large top_k and top_p are.  In registers and histograms a dead token is any bit
// pattern below kEMinBits (kept at or above kDeadBits so that it still has a histogram bin,
// one octave below the live ones, where counts can be checked for completeness); everything
// that weighs or selects tokens looks at patterns >= kEMinBits only.

// Bit pattern of e = 2^(x - M), M = floor(max x) of the row (reference:
// exp2f(x - max) at sampling.cu:235; the common factor 2^(max - M) cancels in
// every probability).  n = floor(x) and f = x - n are exact; 2^f is a degree-5
// Horner polynomial with positive coefficients (monotone, poly(1) < 2); the
// result is scaled by 2^(n - M), n - M <= 0; what falls below 2^-40 is dead
// (kept here as something in [2^-41, 2^-40), see above).
// The significand depends on x alone, so a slice can use its own M and be
// re-based later by an exponent shift.
//
// This is the inner loop of every kernel, and the vector ALU is what bounds
// the streaming pass once the logits arrive fast enough, so the instruction
// count is kept down by hand: the Horner steps with a literal addend are
// written as v_fmaak_f32 (the compiler otherwise spends a move per step on
// some of them), and the scaling is v_cvt_i32_f32 (which saturates) +
// v_ldexp_f32 (exact; anything below 2^-41, zero included, ends at the clamp).
__device__ __forceinline__ uint32_t e_bits_of(float x, float M)
{
    const float n = __builtin_floorf(x);
    const float f = x - n;
    float p = __builtin_fmaf(0x1.e974fap-10f, f, 0x1.277856p-7f);
    asm("v_fmaak_f32 %0, %1, %2, 0x3d648e73" : "=v"(p) : "v"(p), "v"(f));      // p * f + 0x1.c91ce6p-5
    asm("v_fmaak_f32 %0, %1, %2, 0x3e75edab" : "=v"(p) : "v"(p), "v"(f));      // p * f + 0x1.ebdb56p-3
    asm("v_fmaak_f32 %0, %1, %2, 0x3f31725d" : "=v"(p) : "v"(p), "v"(f));      // p * f + 0x1.62e4bap-1
    p = __builtin_fmaf(p, f, 1.0f);
    int k;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(k) : "v"(n - M));
    return __float_as_uint(fmaxf(__builtin_ldexpf(p, k), 0x1p-41f));
}

// The same without the clamp: whatever lies below 2^-40 (zero included) is dead.  For
// code that can tell such tokens by their bin and saves the instruction.
__device__ __forceinline__ uint32_t e_bits_raw(float x, float M)
{
    const float n = __builtin_floorf(x);
    const float f = x - n;
    float p = __builtin_fmaf(0x1.e974fap-10f, f, 0x1.277856p-7f);
    asm("v_fmaak_f32 %0, %1, %2, 0x3d648e73" : "=v"(p) : "v"(p), "v"(f));
    asm("v_fmaak_f32 %0, %1, %2, 0x3e75edab" : "=v"(p) : "v"(p), "v"(f));
    asm("v_fmaak_f32 %0, %1, %2, 0x3f31725d" : "=v"(p) : "v"(p), "v"(f));
    p = __builtin_fmaf(p, f, 1.0f);
    int k;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(k) : "v"(n - M));
    return __float_as_uint(__builtin_ldexpf(p, k));
}

// e of many tokens in one frame: the same bits in eight vector instructions a token instead of ten.
//   * x - floor(x) is one v_fract_f32.  The two differ where x lies in (-2^-25, 0): the subtraction rounds to 1,
//     v_fract stops at 1 - 2^-24 -- and the polynomial is 0x3FFFFFFE, bit for bit, at both.
//   * floor and conversion are one v_cvt_flr_i32_f32 (which saturates, as v_cvt_i32_f32 does).
//   * The frame is in the coefficients, each scaled by 2^-M: a power of two goes through every rounding
//     unchanged while nothing underflows, so |M| <= 100; then the exponent of e needs no subtraction.
// A frame further out is taken off the tokens first (frame_of): x - M is exact for a live token, whose x lies
// within a factor of two of M there, and at most -39 for any token below those.
// Measured: 256 rows of 151936 bfloat16 33.7 -> 32.8 us a call; passes over float32 logits, which wait for memory,
// and the row kernel (tens of instructions a token besides) take what they took.
// The general kernel with penalties keeps e_bits_of: 512 rows of 4096 to 8192 tokens took 2 % longer in this form (22.9 against
// 23.5 us a call, 28.3 against 29.0), and no such call was faster.  Without penalties 1024 rows of 4096 bfloat16 tokens take
// 37.3 us in this form against 39.6.
struct Frame {
    uint32_t c[6];                                       // (uniform: scalar registers)
    __device__ __forceinline__ explicit Frame(int m)
    {
        const uint32_t k[6] = {0x3AF4BA7Du, 0x3C13BC2Bu, 0x3D648E73u, 0x3E75EDABu, 0x3F31725Du, 0x3F800000u};
        const uint32_t d = (uint32_t)__builtin_amdgcn_readfirstlane(m) << 23;
#pragma unroll
        for (int i = 0; i < 6; ++i) c[i] = k[i] - d;
    }
    __device__ __forceinline__ float scaled(float x) const
    {
        int n;
        asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(n) : "v"(x));
        const float f = __builtin_amdgcn_fractf(x);
        float p = __builtin_fmaf(__uint_as_float(c[0]), f, __uint_as_float(c[1]));
#pragma unroll
        for (int i = 2; i < 6; ++i) p = __builtin_fmaf(p, f, __uint_as_float(c[i]));
        return __builtin_ldexpf(p, n);
    }
    // The same, and 0 for x = -inf, whose fractional part v_fract_f32 has as a NaN: its clamp to [0, 1], which makes zeros of NaNs, costs nothing.
    // What x = NaN comes to has no meaning.
    __device__ __forceinline__ float scaled_or_none(float x) const
    {
        int n;
        asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(n) : "v"(x));
        const float f = __builtin_amdgcn_fmed3f(__builtin_amdgcn_fractf(x), 0.0f, 1.0f);
        float p = __builtin_fmaf(__uint_as_float(c[0]), f, __uint_as_float(c[1]));
#pragma unroll
        for (int i = 2; i < 6; ++i) p = __builtin_fmaf(p, f, __uint_as_float(c[i]));
        return __builtin_ldexpf(p, n);
    }
    __device__ __forceinline__ uint32_t raw(float x) const { return __float_as_uint(scaled(x)); }                    // e_bits_raw
    __device__ __forceinline__ uint32_t bits(float x) const { return __float_as_uint(fmaxf(scaled(x), 0x1p-41f)); }  // e_bits_of
};
// The frame of M, the same for all lanes, for the tokens x (bit patterns of floats).
template <int N>
__device__ __forceinline__ Frame frame_of(const float M, uint32_t (&x)[N])
{
    const bool far = __builtin_amdgcn_ballot_w64(!(__builtin_fabsf(M) <= 100.0f)) != 0ull;
    if (__builtin_expect(far, 0)) {
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] = __float_as_uint(fmaxf(__uint_as_float(x[i]) - M, -1000.0f));
    }
    return Frame(far ? 0 : (int)M);
}

// Exact weight of a live token from the bit pattern of e (2^-40 <= e < 2):
// W = e * 2^63 = significand24 << (exponent - 87), in [2^23, 2^64).
__device__ __forceinline__ uint64_t w_of_bits(uint32_t b)
{
    return (uint64_t)((b & 0x7FFFFFu) | 0x800000u) << ((b >> 23) - 87u);
}

// ceil(f * s) for a float 0 < f <= 1 and s < 2^100, exact, clamped to [1, s].
__device__ inline u128 ceil_mul(float f, u128 s)
{
    if (!(f > 0.0f)) return 1;
    if (f >= 1.0f) return s;
    const uint32_t b = __float_as_uint(f);
    int ex = (int)(b >> 23);
    uint64_t m = b & 0x7FFFFFu;
    if (ex == 0) ex = 1; else m |= 0x800000u;
    const int sh = 150 - ex;                                // f = m * 2^-sh, sh >= 24
    u128 r;
    if (sh >= 126) r = 1;                                   // 0 < m*s < 2^124 < 2^sh
    else r = ((u128)m * s + (((u128)1 << sh) - 1)) >> sh;
    if (r < 1) r = 1;
    if (r > s) r = s;
    return r;
}

// 64 random bits -> r in [1, S]: floor(u64 * S / 2^64) + 1
__device__ __forceinline__ u128 r_from_bits(uint64_t u64, u128 S)
{
    const uint64_t s_lo = (uint64_t)S, s_hi = (uint64_t)(S >> 64);
    return (u128)u64 * s_hi + __umul64hi(u64, s_lo) + 1;
}

// floor(a / d) for a < 2^96 and 1 <= d <= 2^20 (a count of tokens), by long division with 32-bit digits.
// Each step divides less than d * 2^32 <= 2^52, which a double holds exactly, by multiplying with 1 / d: off
// by one at most, put right with the remainder.  (The compiler's own 64-bit division takes a few hundred
// dependent instructions per digit.)
__device__ inline u128 div_u32(u128 a, uint32_t d)
{
    const double inv = 1.0 / (double)d;
    uint64_t rem = 0;
    u128 q = 0;
#pragma unroll
    for (int i = 2; i >= 0; --i) {
        const uint64_t cur = (rem << 32) | (uint32_t)(a >> (32 * i));
        uint64_t qi = (uint64_t)((double)cur * inv);
        int64_t r = (int64_t)(cur - qi * d);
        if (r < 0) { qi -= 1u; r += d; }
        if (r >= (int64_t)d) { qi += 1u; r -= d; }
        rem = (uint64_t)r;
        q |= (u128)qi << (32 * i);
    }
    return q;
}

// order-preserving map float -> uint32 (for atomicMax on floats)
__device__ __forceinline__ uint32_t fkey(float x)
{
    const uint32_t b = __float_as_uint(x);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float fkey_inv(uint32_t k)
{
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

// ---------------------------------------------------------- Philox4x32-10 --
// Counter-based generator of Salmon et al.; same stream layout as the
// reference's curand_init(seed, row, 0) (sampling.cu:137): key = seed,
// counter = (draw_lo, draw_hi, row_lo, row_hi).
__device__ inline void philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                     uint32_t k0, uint32_t k1, uint32_t out[4])
{
#pragma unroll
    for (int i = 0; i < 10; ++i) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0;
        const uint32_t n1 = (uint32_t)p1;
        const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1;
        const uint32_t n3 = (uint32_t)p0;
        c0 = n0; c1 = n1; c2 = n2; c3 = n3;
        k0 += 0x9E3779B9u; k1 += 0xBB67AE85u;
    }
    out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}

// ------------------------------------------------------ wave64 primitives --
// All cross-lane traffic uses DPP (data-parallel primitives on the VALU
// operand path): row_shr:1,2,4,8 scan inside each row of 16 lanes, then
// row_bcast:15 carries lane 15 of a row into the next row (rows 1 and 3),
// row_bcast:31 carries lane 31 into rows 2 and 3.  Six steps, no LDS.  Lanes
// with no source read 0 (the identity of + and of max on unsigned).

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp0_u32(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xf, false);
}
template <int CTRL, int ROW_MASK, typename T>
__device__ __forceinline__ T dpp0(T v)
{
    static_assert(sizeof(T) == 4 || sizeof(T) == 8, "32- or 64-bit integers (128-bit sums have scans of their own below)");
    if constexpr (sizeof(T) == 4) return (T)dpp0_u32<CTRL, ROW_MASK>((uint32_t)v);
    else {
        const uint32_t lo = dpp0_u32<CTRL, ROW_MASK>((uint32_t)v), hi = dpp0_u32<CTRL, ROW_MASK>((uint32_t)((uint64_t)v >> 32));
        return (T)(((uint64_t)hi << 32) | lo);
    }
}

// Inclusive scan (sum) over the 64 lanes; lane 63 ends with the wave total.
// The reference's float ladder has to run 16,8,4,2,1 to stay monotone
// (sampling.cu:48-58); these are integers, exact in any order.
template <typename T>
__device__ __forceinline__ T wave_inclusive_scan(T v)
{
    v += dpp0<0x111, 0xf>(v);     // row_shr:1
    v += dpp0<0x112, 0xf>(v);     // row_shr:2
    v += dpp0<0x114, 0xf>(v);     // row_shr:4
    v += dpp0<0x118, 0xf>(v);     // row_shr:8
    v += dpp0<0x142, 0xa>(v);     // row_bcast:15 -> rows 1,3
    v += dpp0<0x143, 0xc>(v);     // row_bcast:31 -> rows 2,3
    return v;
}

__device__ __forceinline__ uint32_t lane63_u32(uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, 63); }
template <typename T>
__device__ __forceinline__ T lane63(T v)
{
    if constexpr (sizeof(T) == 4) return (T)lane63_u32((uint32_t)v);
    else if constexpr (sizeof(T) == 8) return (T)(((uint64_t)lane63_u32((uint32_t)((uint64_t)v >> 32)) << 32) | lane63_u32((uint32_t)v));
    else return (T)(((u128)lane63((uint64_t)((u128)v >> 64)) << 64) | lane63((uint64_t)v));
}

// Sum over the wave, returned to every lane (wave-uniform).
template <typename T>
__device__ __forceinline__ T wave_sum(T v) { return lane63(wave_inclusive_scan(v)); }

__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v)
{
    v = max(v, dpp0_u32<0x111, 0xf>(v));
    v = max(v, dpp0_u32<0x112, 0xf>(v));
    v = max(v, dpp0_u32<0x114, 0xf>(v));
    v = max(v, dpp0_u32<0x118, 0xf>(v));
    v = max(v, dpp0_u32<0x142, 0xa>(v));
    v = max(v, dpp0_u32<0x143, 0xc>(v));
    return lane63_u32(v);
}

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

// A mass as four limbs of 24 bits in 32-bit words: sums of up to 256 of them need no carries, so a scan
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

// 128-bit sums of masses (a row's total stays below 2^84) go the same way.
__device__ __forceinline__ u128 wave_inclusive_scan(u128 v) { return wide(m96(wave_inclusive_scan(limbs(m96(v))))); }
__device__ __forceinline__ u128 wave_sum(u128 v) { return wide(m96(lane_of(wave_inclusive_scan(limbs(m96(v))), 63u))); }

}  // namespace rs
