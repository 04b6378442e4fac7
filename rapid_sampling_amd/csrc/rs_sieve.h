// The sieve path: one pass over the logits in which every wave works a slice of its own, a finishing workgroup per row.
#pragma once

#include "rs_common.h"
#include "rs_mass.h"
#include "rs_sieve_view.h"
#include "rs_stream.h"

namespace rs {

// ---------------------------------------------------------------- sieve path --
// For kept sets that are small next to the row two things are needed of it: its largest tokens, and its total mass D, of
// which P = ceil(top_p * D) is the mass that is enough.  The tokens must be exact.  D need not be, as long as the token that is
// picked with it is the one that every D within its error picks: then the exact D picks it, too.  So
//
//   sieve_kernel         a workgroup per slice, no histogram, two barriers.  It sums 2^x with the hardware's exponential and sets aside every token at
//                        or above a value that a given number of its threads, pair by pair, reach with their largest token: between that
//                        many and some half more, whatever the distribution.
//   sieve_finish_kernel  a workgroup per row.  It takes D from the slices' sums, works out threshold and token from the tokens set
//                        aside -- complete above the largest of the slices' bounds -- and then compares the target's distance from
//                        both ends of the token's place with what the error of D can shift them by.  If it is too close (a row in a million for
//                        each token kept) it sums the row again, from the logits, in double precision, and decides again; exactly, when that
//                        is too close as well.
//
// The results are the same integers as on every other path.
//
// The error of D, in units of 2^-24 of it: v_exp_f32(x) is larger than e of x by -2.96 to 3.45 (a test compares every float); 16 tokens are
// summed in a tree of four roundings, of one unit each at most, their sums in double precision, and the slice's sum is rounded once to a float, one more:
// 8.45, for which 9 are allowed.  The slices' are added as integers of 2^-40 of the frame, cut off, which is less than what is allowed for the tokens of no
// weight (below).  A wave with a value out of v_exp_f32's range, or with a NaN or an infinity, sums 2^(x - M), M the floor of its maximum, whose x - M is
// rounded: |v_exp_f32(x - M) / e - 1| is at most 5.9 units for tokens up to 8 octaves below the frame, 8.7 to 16, 14.1 to 32, 25.5 to 40 (the same test; where
// |x| is 128 and more, x - M is exact), so for 4096 tokens, one of them in the frame's octave, at most 9; with 3 roundings 12, and 32
// are allowed.  Tokens more than 40 octaves below the row's frame weigh nothing but are in the sums: 2^-40 each at most.
//
// Where the pass waits for the memory (the host's rule) it sums the tokens' own e in double precision instead (FINE): 2^-40 of D and of the slices' number
// is allowed for, and the tokens of no weight only if the least token of a slice is that far down.  Then hardly a row is summed again.  (Logits of -inf
// must not make a wave one that is out of range: 128 x 262144 with penalties and one logit in twenty -inf 94.7 us a call, 59.3 as it is; 128 x 1048576
// N(0,3), top_k 1000, top_p 0.3, some of whose rows were then summed again, 327.)
// What was summed in a frame counts only where it weighs: not in a wave or a slice all of whose tokens are 41 octaves down, a masked stretch.
//
// What bounds it: in large calls of float32 the read: 128 rows of 1048576 take 93 to 99 us a pass on average (86 at the fastest), a kernel that only reads them 81
// to 87; there a token costs some 20 vector instructions (FINE).  Without that it costs 4.6 (one of them the exponential, 2.7 issue slots) and a wave some 200
// for bound and staging, some 10 a token together, where the pass with exact e and a histogram (stream_kernel) takes 22 and an LDS atomic.  us of a pass,
// there / here: 128 rows of 1048576 112 / 93 to 99, 64 of 152064 12.7 / 10.4, 256 of 151936 bfloat16 28 / 17, of which 12 are the read.
constexpr uint32_t kSieveErrOdd = 19;                    // D is known to 2^-19 of itself when waves were summed in a frame, else to 9 * 2^-24

// Sum over the wave in double precision, in every lane.
__device__ __forceinline__ double wave_sum_f64(double v)
{
    auto step = [&](auto ctrl, auto mask) {
        v += __builtin_bit_cast(double, dpp0<decltype(ctrl)::value, decltype(mask)::value>(__builtin_bit_cast(uint64_t, v)));
    };
    step(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{}); step(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{}); step(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{}); step(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});
    return __builtin_bit_cast(double, lane63(__builtin_bit_cast(uint64_t, v)));
}

struct LdsSieve {
    float4   grp[kWaves][kWave];                         // groups of four tokens that hold one to set aside
    uint32_t gidx[kWaves][kWave];
    double   mass[kThreads];                             // the threads' sums
    float    top[kThreads];                              // and largest tokens
    float    frame[kWaves];                              // the frames of the sums
    uint32_t wmax[kWaves], odd[kWaves], n[2][kWaves], low[kWaves], tie;
};

// A workgroup's slice to its record.  group(j, x): the scaled logits of the thread's j-th group of four tokens, group j * 256 + tid of the
// slice, from the registers that the loads fill; those past the end of the row, `left` groups from the slice's first, are copies of its last;
// strange(): the thread has seen input that must be cleaned up; redo(j, x): the group again, cleaned up; then(): behind the last of these;
// g0: the slice's first group.
// The terms of the sum need no frame: 2^x is a float for every x in question, and so they are worked out in the order in which
// the loads arrive.  A wave whose largest x is beyond 120 or below -80 (the tokens 40 octaves below it would no longer be floats), or
// that holds a NaN or an infinity, does it again, cleaned up and in a frame.
//
// kGrain: two tokens' keys are equal or further apart than this.  Halving a range ends there: 10 turns less for bfloat16, whose ties hardly ever leave as many
// threads as are wanted (512 x 32768 with logits near 20, top_k 50: 29.7 us a call with 1, 26.7 like this).
constexpr uint32_t sieve_grain(int dtype) { return dtype == RS_DTYPE_BF16 ? 1u << 13 : dtype == RS_DTYPE_F16 ? 1u << 10 : 1u; }   // (of products of 8 and 11 bits by one factor)
template <int R, bool FINE, uint32_t kGrain, typename G, typename Z, typename A, typename E>
__device__ __forceinline__ void sieve_slice(const SieveView &v, LdsSieve &s, G group, Z strange, A redo, E then, const size_t slice, const uint32_t g0, const uint32_t left, const int tid)
{
    const float kInf = __builtin_inff();
    const int lane = tid & (kWave - 1), wave = (int)uniform((uint32_t)tid >> 6);
    bool odd = false;
    double mass = 0.0;
    const Frame fr(0);
    float low = kInf;                                    // FINE: the smallest, or a NaN if there is one
    float x[R * 4], gm[R], lm = -kInf, M = 0.0f;            // gm: the largest of every group, lm: of all; of the wave: the frame, the sum in it
    auto top = [&](int j) {
        float m;                                         // (fmaxf quiets its operands first, an instruction each; products are quiet)
        asm("v_max3_f32 %0, %1, %2, %3" : "=v"(m) : "v"(x[j * 4]), "v"(x[j * 4 + 1]), "v"(x[j * 4 + 2]));
        asm("v_max_f32 %0, %1, %2" : "=v"(m) : "v"(m), "v"(x[j * 4 + 3]));
        return m;
    };
    if ((uint32_t)(wave * kWave) >= left) {              // nothing of the row
#pragma unroll
        for (int j = 0; j < R; ++j) gm[j] = -kInf;
    } else {
        const bool ragged = left < (uint32_t)(R * kThreads);             // some of the groups may lie past the end of the row
        float part[R / 4], q[4];                         // (a tree: log2 of the tokens' number of roundings)
#pragma unroll
        for (int j = 0; j < R; ++j) {
            group(j, &x[j * 4]);
            gm[j] = top(j);
            if constexpr (FINE) {
                float least;                             // (see top)
                asm("v_minimum3_f32 %0, %1, %2, %3" : "=v"(least) : "v"(x[j * 4]), "v"(x[j * 4 + 1]), "v"(x[j * 4 + 2]));
                asm("v_minimum3_f32 %0, %1, %2, %3" : "=v"(low) : "v"(least), "v"(x[j * 4 + 3]), "v"(low));
                const bool in = !ragged || (uint32_t)(j * kThreads) + opaque((uint32_t)tid) < left;
                auto e = [&](int q) { return (double)fr.scaled_or_none(x[j * 4 + q]); };
                const double d0 = e(0) + e(1), d1 = e(2) + e(3);
                mass += in ? d0 + d1 : 0.0;
                q[j % 4] = 0.0f;
            } else
                q[j % 4] = (__builtin_amdgcn_exp2f(x[j * 4]) + __builtin_amdgcn_exp2f(x[j * 4 + 1])) +
                           (__builtin_amdgcn_exp2f(x[j * 4 + 2]) + __builtin_amdgcn_exp2f(x[j * 4 + 3]));
            if (j % 2 == 1) {
                if (ragged) {
                    const uint32_t at = (uint32_t)((j - 1) * kThreads) + opaque((uint32_t)tid);
                    if (at >= left) { gm[j - 1] = -kInf; q[j % 4 - 1] = 0.0f; }
                    if (at + (uint32_t)kThreads >= left) { gm[j] = -kInf; q[j % 4] = 0.0f; }
                }
                lm = fmaxf(fmaxf(lm, gm[j - 1]), gm[j]);
                __builtin_amdgcn_sched_barrier(0);       // (group after group, as they arrive: side by side they would take 30 registers more)
            }
            if (j % 4 == 3) part[j / 4] = (q[0] + q[1]) + (q[2] + q[3]);
        }
        if constexpr (!FINE) {
#pragma unroll
            for (int i = 0; i < R / 4; ++i) mass += (double)part[i];
        }
        odd = __builtin_amdgcn_ballot_w64(!(mass < (double)kInf) || lm > 120.0f || (FINE && low != low) || strange()) != 0ull || __builtin_amdgcn_ballot_w64(lm >= -80.0f) == 0ull;
        if (__builtin_expect(odd, 0)) {
            const uint32_t t = opaque((uint32_t)tid);
            lm = -kInf;
#pragma unroll
            for (int j = 0; j < R; ++j) {
                redo(j, &x[j * 4]);
                gm[j] = (uint32_t)(j * kThreads) + t < left ? top(j) : -kInf;
                lm = fmaxf(lm, gm[j]);
            }
            M = __builtin_floorf(fkey_inv(wave_max_u32(fkey(lm))));
            mass = 0.0;
#pragma unroll
            for (int j = 0; j < R; ++j) {
                auto e = [&](int q) { return __builtin_amdgcn_exp2f(x[j * 4 + q] - M); };
                mass += (uint32_t)(j * kThreads) + t < left ? (double)((e(0) + e(1)) + (e(2) + e(3))) : 0.0;
            }
        }
    }
    then();
    s.top[tid] = lm; s.mass[tid] = mass;
    {
        const uint32_t k = wave_max_u32(fkey(lm));
        if (lane == 0) { s.frame[wave] = M; s.wmax[wave] = k; s.odd[wave] = odd ? 1u : 0u; }
        if constexpr (FINE) {
            const uint32_t l = wave_max_u32(~fkey(low));
            if (lane == 0) s.low[wave] = l;
        }
    }
    if (tid == 0) s.tie = 1u;
    __syncthreads();

    // The bound: a value that at least `reach` of 128 pairs of threads reach with their largest token, and not many more, by halving
    // the range of these (of their order-preserving keys: on scalars).  Every wave for itself.  (Tokens 41 octaves below the slice's frame
    // are dead wherever the row's frame is.)
    const float4 t4 = reinterpret_cast<const float4 *>(s.top)[lane];
    const uint4 k4 = *reinterpret_cast<const uint4 *>(s.wmax);
    const uint32_t one = fkey(fmaxf(t4.x, t4.y)), two = fkey(fmaxf(t4.z, t4.w));
    const uint32_t key = uniform(max(max(k4.x, k4.y), max(k4.z, k4.w)));
    const float xmax = fkey_inv(key), Ms = __builtin_floorf(xmax);
    auto reached = [&](uint32_t t) {
        return (uint32_t)(__builtin_popcountll(__builtin_amdgcn_ballot_w64(one >= t)) + __builtin_popcountll(__builtin_amdgcn_ballot_w64(two >= t)));
    };
    uint32_t want = v.reach, hi = key;
    const uint32_t dead = uniform(fkey(Ms - 41.0f));
    // (from the least of a few of them, which is below the bound nearly always; else from the least of all)
    uint32_t lo = max(min(min(lane_of(one, 0u), lane_of(two, 16u)), min(lane_of(one, 32u), lane_of(two, 48u))), dead), reach = reached(lo);
    if (reach < want) { lo = max(~wave_max_u32(~min(one, two)), dead); reach = reached(lo); }
    const uint32_t room = v.units * (uint32_t)kWave;
    bool full = false;
    float bound = 0.0f;
    uint32_t c[kWaves] = {0u, 0u, 0u, 0u};               // of each wave, its groups that reach the bound
    for (uint32_t turn = 0;; turn ^= 1u) {
#pragma unroll 1
        while (reach > want + 3u && hi - lo > kGrain) {
            const uint32_t mid = lo + ((hi - lo) >> 1), r = reached(mid);
            if (r >= want) { lo = mid; reach = r; } else hi = mid;
        }
        // (ties at the bound, of more threads than there is room for: none of them)
        auto leave_ties = [&]() { lo = hi; hi = key; reach = want = reached(lo); };
        if (__builtin_expect(hi - lo <= kGrain && lo != key && reach * 2u > room, 0)) {
            const float4 t = reinterpret_cast<const float4 *>(s.top)[opaque((uint32_t)lane)];            // (again: kept, it would cost the usual way registers)
            uint32_t threads = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) threads += (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(fkey(i == 0 ? t.x : i == 1 ? t.y : i == 2 ? t.z : t.w) >= lo));
            if (threads > room) leave_ties();
        }
        bound = fkey_inv(lo);
        // the wave's groups that reach it, side by side
        uint32_t fill = 0;
        const uint32_t first = opaque(g0 + (uint32_t)tid);          // (or sixteen sums of it are kept from the loads on)
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const bool in = gm[j] >= bound;
            const uint64_t vote = __builtin_amdgcn_ballot_w64(in);
            if (vote != 0ull) {
                const uint32_t at = fill + __builtin_amdgcn_mbcnt_hi((uint32_t)(vote >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)vote, 0u));
                if (in && at < (uint32_t)kWave) {
                    s.grp[wave][at] = make_float4(x[j * 4], x[j * 4 + 1], x[j * 4 + 2], x[j * 4 + 3]);
                    s.gidx[wave][at] = first + (uint32_t)(j * kThreads);
                }
                fill += (uint32_t)__builtin_popcountll(vote);
            }
        }
        if (lane == 0) s.n[turn][wave] = fill;
        __syncthreads();
        const uint4 f4 = *reinterpret_cast<const uint4 *>(s.n[turn]);
        c[0] = uniform(f4.x); c[1] = uniform(f4.y); c[2] = uniform(f4.z); c[3] = uniform(f4.w);
        const uint32_t most = max(max(c[0], c[1]), max(c[2], c[3]));
        if (__builtin_expect(most <= (uint32_t)kWave && c[0] + c[1] + c[2] + c[3] <= room, 1)) break;
        // more groups than there is room for (threads with many of them, ties): fewer threads, in the end one; if there are too many like it, none
        if (want == 1u || lo == key) { full = true; break; }
        if (hi - lo <= kGrain) leave_ties();
        else { want = want > 8u ? want - 8u : 1u; hi = key; }
    }
    if (wave == 1) {
        // the slice's sum: lane l those of threads 4 l to 4 l + 3, all of one wave
        const double2 m2 = reinterpret_cast<const double2 *>(s.mass)[lane * 2], m3 = reinterpret_cast<const double2 *>(s.mass)[lane * 2 + 1];
        const int down = (int)fmaxf(s.frame[lane >> 4] - Ms, -1000.0f);
        const double all = wave_sum_f64(__builtin_ldexp((m2.x + m2.y) + (m3.x + m3.y), down));
        const uint4 o4 = *reinterpret_cast<const uint4 *>(s.odd);
        const uint32_t odds = uniform(o4.x | o4.y | o4.z | o4.w);
        bool any = false;
        if (__builtin_expect(odds != 0u, 0)) {
            const float4 m4 = *reinterpret_cast<const float4 *>(s.frame);
            const float from = Ms - 41.0f;
            any = (o4.x != 0u && m4.x >= from) || (o4.y != 0u && m4.y >= from) || (o4.z != 0u && m4.z >= from) || (o4.w != 0u && m4.w >= from);
        }
        if (lane == 0) {
            v.hdr[slice].mass = __float_as_uint((float)all) | (any ? kSieveOdd : 0u);
            if constexpr (FINE) {                        // (a wave that was cleaned up may hold anything: -inf)
                const uint32_t low = odds != 0u ? 0x007FFFFFu : ~max(max(s.low[0], s.low[1]), max(s.low[2], s.low[3]));
                v.fine[slice] = SieveFine{all, low, 0u};
            }
        }
    }
    uint32_t n = 0, cut = key;
    if (__builtin_expect(full, 0)) {
        float least = xmax;
        const uint32_t t0 = opaque((uint32_t)tid);
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const float m = fminf(fminf(x[j * 4], x[j * 4 + 1]), fminf(x[j * 4 + 2], x[j * 4 + 3]));
            if ((uint32_t)(j * kThreads) + t0 < left) least = fminf(least, m);
        }
        if (least != xmax) s.tie = 0u;
        __syncthreads();
        n = s.tie ? kSieveTie : 0u;
    } else if (wave == 0) {
        // the tokens of those groups, by the first wave, a group to a lane
        const uint32_t all = c[0] + c[1] + c[2] + c[3];
        uint64_t *st = v.stash + slice * room;
        // the group that is the lane's u-th
        auto group_of = [&](const uint32_t g, float (&t)[4]) __attribute__((always_inline)) {
            uint32_t w = 0, at = g;
            if (at >= c[0]) { at -= c[0]; w = 1u; }
            if (w == 1u && at >= c[1]) { at -= c[1]; w = 2u; }
            if (w == 2u && at >= c[2]) { at -= c[2]; w = 3u; }
            const float4 q4 = s.grp[w][at & 63u];
            t[0] = q4.x; t[1] = q4.y; t[2] = q4.z; t[3] = q4.w;
            return s.gidx[w][at & 63u] * 4u;
        };
        for (;;) {
            n = 0;
            for (uint32_t g = (uint32_t)lane; g < room; g += kWave) {
                const bool have = g < all;
                float t[4];
                const uint32_t i0 = group_of(g, t);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const bool in = have && t[q] >= bound;
                    const uint64_t vote = __builtin_amdgcn_ballot_w64(in);
                    const uint32_t o = n + __builtin_amdgcn_mbcnt_hi((uint32_t)(vote >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)vote, 0u));
                    if (in && o < room) st[o] = ((uint64_t)__float_as_uint(t[q]) << 32) | (i0 + (uint32_t)q);
                    n += (uint32_t)__builtin_popcountll(vote);
                }
            }
            if (__builtin_expect(n <= room, 1)) { cut = lo - 1u; break; }
            // Too many (several tokens of a group): a bound is looked for that no more reach than there is room for, but v.keep all the same, or as many as ties
            // leave -- upwards in steps of a 64th to a 32nd of it, twice as long each time, until they fit, then by halving.  Too many reach `over`, from
            // `fits` on they fit.  (A fixed part of the way up to the slice's largest token depends on how far up that is: in rows with a few spikes hardly a
            // token was left, and rows whose top_k tokens were then not all there had to be summed again, 64 x 1048576 with a top_k of 1024 455 us a call,
            // 59 like this.  There is always a slice like that in a call of hundreds: what this takes the whole call takes longer.)
            uint32_t k8[8];
#pragma unroll
            for (uint32_t u = 0; u < 2u; ++u) {
                const uint32_t g = u * kWave + (uint32_t)lane;
                float t[4];
                group_of(g, t);
#pragma unroll
                for (int q = 0; q < 4; ++q) k8[u * 4u + q] = g < all ? fkey(t[q]) : 0u;
            }
            uint32_t over = lo, fits = key + 1u;
            auto next_to = [&](const uint32_t k) __attribute__((always_inline)) {        // the least token's key from k on, all ones if there is none
                uint32_t least = ~0u;
#pragma unroll
                for (int i = 0; i < 8; ++i) least = k8[i] >= k ? min(least, k8[i]) : least;
                return ~wave_max_u32(~least);
            };
            auto reach_it = [&](const uint32_t k) __attribute__((always_inline)) {
                uint32_t r = 0;
#pragma unroll
                for (int i = 0; i < 8; ++i) r += (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(k8[i] >= k));
                return r;
            };
            // (past the least token's value first: there may be many of it)
            const uint32_t next = next_to(next_to(lo) + 1u);
            if (next <= key) {
                if (reach_it(next) <= room) over = (fits = next) - 1u; else over = next;
            } else over = key;
            for (uint32_t step = 1u << 18; fits - over > 1u; step *= 2u) {
                const uint32_t mid = fits <= key ? over + ((fits - over) >> 1) : key - over > step ? over + step : key, r = reach_it(mid);
                if (r > room) over = mid;
                else { fits = mid; if (r >= v.keep) break; }
            }
            if (fits > key) { n = 0; break; }            // ties of the largest
            lo = fits; bound = fkey_inv(lo);
        }
    }
    if (tid == 0) {
        *reinterpret_cast<uint2 *>(&v.hdr[slice]) = make_uint2(key, n);
        v.hdr[slice].cut = cut;
    }
}

// A workgroup of 256 threads to a slice of R * 256 groups of four tokens.
template <int R, int DT, bool FINE>
__global__ void __launch_bounds__(kThreads, R == 16 ? (FINE ? 3 : 4) : !FINE ? 8 : R == 8 ? 5 : 8) sieve_kernel(const Params p, const SieveView v)
{
    __shared__ LdsSieve s;
    const int tid = threadIdx.x;
    const uint32_t row = blockIdx.x / v.G, part = blockIdx.x - row * v.G;
    const bool reporter = blockIdx.x == 0 && tid == 0;
    PrevCall prev;
    prev.slow_rows = 0; prev.meta = 0;
    if (reporter) prev = report_begin(p);
    const uint32_t g0 = part * (uint32_t)(R * kThreads), left = ((uint32_t)p.V >> 2) - g0;
    // the thread's j-th group is group j * 256 + tid; past the end of the row its last one
    typedef typename std::conditional<DT == RS_DTYPE_F32, rs_u32x4, rs_u32x2>::type T;
    typedef const __attribute__((address_space(1))) T GlobalT;
    GlobalT *from = (GlobalT *)reinterpret_cast<const T *>(logits_row(p, row)) + g0;
    T l[R];
    if (left >= (uint32_t)(R * kThreads)) {              // (a scalar address and the thread's offset: none is worked out per thread)
#pragma unroll
        for (int j = 0; j < R; ++j) {
            GlobalT *q = from + j * kThreads;
            asm("" : "+s"(q));
            l[j] = __builtin_nontemporal_load(q + (uint32_t)tid);
        }
    } else {
#pragma unroll
        for (int j = 0; j < R; ++j) l[j] = __builtin_nontemporal_load(from + min((uint32_t)(j * kThreads + tid), left - 1u));
    }
    if (reporter) report_end(p, prev, true);
    sieve_slice<R, FINE, sieve_grain(DT)>(v, s, [&](int j, float *x) {
        uint32_t w[4];
        if constexpr (DT == RS_DTYPE_F32) { w[0] = l[j].x; w[1] = l[j].y; w[2] = l[j].z; w[3] = l[j].w; }
        else widen4(make_uint2(l[j].x, l[j].y), DT, w);
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = __uint_as_float(w[q]) * p.c;
    }, [] { return false; }, [](int, float *x) {
        // (the clean-up of sampling.cu:553 on the products in the registers)
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = sf(x[q]);
    }, [] {}, (size_t)row * v.G + part, g0, left, tid);
}

// The same with penalties: x = sf((sf(l) - pen) * c) (sampling.cu:220).  The pass also writes what every penalty will be unless its token is
// sampled, fma(pen, decay, 0), and sieve_pen_fix_kernel patches the sampled token's once it is known.  Penalties are non-zero only
// where tokens have been generated, and a finite decay leaves +0.0 as it is: so a wave lists its groups with a bit set in one of their penalties, in
// LDS, and writes from the list: the new values where they belong, the old ones into its notes, from which the sampled token's is looked up and a
// row that must be read again gets its old values back.  A wave with more such groups than the list takes leaves its penalties to the fix-up kernel
// and says so.
//
// What bounds it: the memory.  128 x 262144 tokens, two in a hundred penalised, inputs from HBM: 65.5 us, of which 50 are the read (the writes left out
// of a copy of it) and 15 the lines of the penalties that change, half of all lines; written in whole groups of 64 or 128 bytes 65.0 and 68.5, with
// non-temporal stores 67.0, with slices of 4096 tokens 66.0.  The pass with a histogram and a vote about every single penalty (stream_pen_kernel), 35
// vector instructions a token, takes 74.
template <int R, int DT, bool FINE>
__global__ void __launch_bounds__(kThreads, R == 8 ? 4 : 6) sieve_pen_kernel(const Params p, const SieveView v)
{
    constexpr uint32_t kCap = sieve_pen_cap(R);
    __shared__ LdsSieve s;
    __shared__ float4 old[kWaves][kCap];
    __shared__ uint32_t at[kWaves][kCap];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = (int)uniform((uint32_t)tid >> 6);
    const uint32_t row = blockIdx.x / v.G, part = blockIdx.x - row * v.G;
    const bool reporter = blockIdx.x == 0 && tid == 0;
    PrevCall prev;
    prev.slow_rows = 0; prev.meta = 0;
    if (reporter) prev = report_begin(p);
    const uint32_t g0 = part * (uint32_t)(R * kThreads), left = ((uint32_t)p.V >> 2) - g0;
    typedef typename std::conditional<DT == RS_DTYPE_F32, rs_u32x4, rs_u32x2>::type T;
    typedef const __attribute__((address_space(1))) T GlobalT;
    typedef const __attribute__((address_space(1))) rs_u32x4 GlobalP;
    GlobalT *from = (GlobalT *)reinterpret_cast<const T *>(logits_row(p, row)) + g0;
    rs_u32x4 *pens = reinterpret_cast<rs_u32x4 *>(p.penalties + (int64_t)row * p.V) + g0;
    GlobalP *pfrom = (GlobalP *)pens;
    const bool ragged = left < (uint32_t)(R * kThreads);
    T l[R];
    rs_u32x4 pn[R];
    if (!ragged) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
            GlobalT *q = from + j * kThreads;
            GlobalP *b = pfrom + j * kThreads;
            asm("" : "+s"(q), "+s"(b));
            l[j] = __builtin_nontemporal_load(q + (uint32_t)tid);
            pn[j] = b[(uint32_t)tid];
        }
    } else {
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const uint32_t i = min((uint32_t)(j * kThreads + tid), left - 1u);
            l[j] = __builtin_nontemporal_load(from + i);
            pn[j] = pfrom[i];
        }
    }
    if (reporter) report_end(p, prev, true);
    const size_t slice = (size_t)row * v.G + part;
    auto widen = [&](const T &t, uint32_t (&w)[4]) __attribute__((always_inline)) {
        if constexpr (DT == RS_DTYPE_F32) { w[0] = t.x; w[1] = t.y; w[2] = t.z; w[3] = t.w; }
        else widen4(make_uint2(t.x, t.y), DT, w);
    };
    uint32_t fill = 0;
    uint32_t low = 0u;                                   // bit pattern of the most negative penalty
    sieve_slice<R, FINE, 1u>(v, s, [&](int j, float *x) __attribute__((always_inline)) {
        uint32_t w[4];
        widen(l[j], w);
        const uint32_t b[4] = {pn[j].x, pn[j].y, pn[j].z, pn[j].w};
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = (__uint_as_float(w[q]) - __uint_as_float(b[q])) * p.c;
        bool any = ((b[0] | b[1] | b[2]) | b[3]) != 0u;
        if (ragged) any = any && (uint32_t)(j * kThreads) + opaque((uint32_t)tid) < left;
        const uint64_t vote = __builtin_amdgcn_ballot_w64(any);
        if (vote != 0ull) {
            const uint32_t o = fill + __builtin_amdgcn_mbcnt_hi((uint32_t)(vote >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)vote, 0u));
            if (any && o < kCap) {
                old[wave][o] = make_float4(__uint_as_float(b[0]), __uint_as_float(b[1]), __uint_as_float(b[2]), __uint_as_float(b[3]));
                at[wave][o] = (uint32_t)(j * kThreads + tid);
            }
            fill += (uint32_t)__builtin_popcountll(vote);
            // (a logit of -inf is the lowest float before the penalty is taken off: only with a penalty of its size, here -1e30, does it matter)
            low = max(low, max(max(b[0], b[1]), max(b[2], b[3])));
        }
    }, [&] { return low > 0xF149F2CAu; }, [&](int j, float *x) __attribute__((always_inline)) {
        const uint32_t i = min((uint32_t)(j * kThreads) + opaque((uint32_t)tid), left - 1u);
        uint32_t w[4];
        const T t = from[i];
        widen(t, w);
        const rs_u32x4 q4 = pfrom[i];
        const uint32_t b[4] = {q4.x, q4.y, q4.z, q4.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = sf((sf(__uint_as_float(w[q])) - __uint_as_float(b[q])) * p.c);
    }, [&]() __attribute__((always_inline)) {
        const size_t mine = slice * kWaves + (size_t)wave;
        const bool fits = fill <= kCap;
        if (lane == 0) v.noted[mine] = fits ? fill : kSievePenLeft;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (fits)
            for (uint32_t i = (uint32_t)lane; i < fill; i += kWave) {
                const float4 q = old[wave][i];
                const uint32_t g = at[wave][i];
                v.note_at[mine * kCap + i] = g0 + g;
                v.note_old[mine * kCap + i] = q;
                reinterpret_cast<float4 *>(pens)[g] = make_float4(__builtin_fmaf(q.x, p.decay, 0.0f), __builtin_fmaf(q.y, p.decay, 0.0f),
                                                                  __builtin_fmaf(q.z, p.decay, 0.0f), __builtin_fmaf(q.w, p.decay, 0.0f));
            }
    }, slice, g0, left, tid);
}

// The sampled token's penalty, pen <- fma(pen, decay, pen == 0 ? presence : repetition) (sampling.cu:427-437), the old value from the notes
// (+0.0 when its group is not among them), and all penalties of the waves that left theirs.  v.fixers workgroups to a row, each for every
// v.fixers-th slice, wave w for wave w's part of them: mostly it is one look at some words and a chain of two loads for the one token (4.7 us
// behind 128 x 262144 tokens, with 2, 8 or 32 workgroups to a row alike; but rows of nothing but non-zero penalties
// pay for every slice that a workgroup does after another: 64 x 50304 21.9 us a call with 8, 17.7 with 32).
template <int R>
__global__ void __launch_bounds__(kThreads) sieve_pen_fix_kernel(const Params p, const SieveView v)
{
    constexpr uint32_t kCap = sieve_pen_cap(R);
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = (int)uniform((uint32_t)tid >> 6);
    const uint32_t row = blockIdx.x / v.fixers, first = blockIdx.x - row * v.fixers, G = v.G;
    const uint32_t part = first + (uint32_t)lane * v.fixers;         // the lane's slice (64 of them at most)
    const uint32_t *noted = v.noted + (size_t)row * G * kWaves;
    const uint32_t n = noted[min(part, G - 1u) * (uint32_t)kWaves + (uint32_t)wave], token = uniform((uint32_t)p.out[row]);
    const uint32_t V4 = (uint32_t)p.V >> 2, group = token >> 2;
    float *pens = p.penalties + (int64_t)row * p.V;
    uint64_t to_do = __builtin_amdgcn_ballot_w64(part < G && n == kSievePenLeft);
    // the sampled token's slice, if it is one of this workgroup's and its group this wave's, and the penalties have been written
    const uint32_t its = group / (uint32_t)(R * kThreads), l = its / v.fixers;
    if (token < (uint32_t)p.V && its - l * v.fixers == first && ((group >> 6) & (uint32_t)(kWaves - 1)) == (uint32_t)wave && !(to_do >> l & 1ull)) {
        const size_t rec = (((size_t)row * G + its) * kWaves + (size_t)wave) * kCap;
        const uint32_t have = min(lane_of(n, l), kCap);
        constexpr uint32_t kLooks = (kCap + kWave - 1u) / kWave;
        uint32_t is[kLooks];
        float old[kLooks], o = 0.0f;                     // (asked for before it is known which: a chain of two loads, not of three)
        bool mine = false;
#pragma unroll
        for (uint32_t u = 0; u < kLooks; ++u) {
            const size_t i = rec + min(u * kWave + (uint32_t)lane, kCap - 1u);
            is[u] = v.note_at[i]; old[u] = reinterpret_cast<const float *>(&v.note_old[i])[token & 3u];
        }
#pragma unroll
        for (uint32_t u = 0; u < kLooks; ++u)
            if (u * kWave + (uint32_t)lane < have && is[u] == group) { o = old[u]; mine = true; }
        const uint64_t found = __builtin_amdgcn_ballot_w64(mine);
        if (found ? mine : lane == 0) pens[token] = __builtin_fmaf(o, p.decay, o == 0.0f ? p.presence : p.repetition);
    }
    while (to_do) {
        const uint32_t at = first + (uint32_t)__builtin_ctzll(to_do) * v.fixers;
        to_do &= to_do - 1ull;
        float4 w[R];
        uint32_t g[R];
#pragma unroll
        for (int j = 0; j < R; ++j) {
            g[j] = at * (uint32_t)(R * kThreads) + (uint32_t)(j * kThreads + tid);
            w[j] = reinterpret_cast<const float4 *>(pens)[min(g[j], V4 - 1u)];
        }
#pragma unroll
        for (int j = 0; j < R; ++j)
            if (g[j] < V4) {
                auto next = [&](float o, uint32_t i) { return __builtin_fmaf(o, p.decay, g[j] * 4u + i != token ? 0.0f : o == 0.0f ? p.presence : p.repetition); };
                reinterpret_cast<float4 *>(pens)[g[j]] = make_float4(next(w[j].x, 0u), next(w[j].y, 1u), next(w[j].z, 2u), next(w[j].w, 3u));
            }
    }
}

// ---- the finish ----
constexpr uint32_t kSieveList = 2048;                    // tokens at or above the boundary bin that are listed at most
constexpr int      kSieveCopies = 4;                     // of each level-1 bin while it is counted
constexpr uint32_t kSieveSteps = 256;                    // between the bound and the row's largest token, where the short way counts
template <int NT>
struct LdsSieveFin {
    alignas(16) uint64_t bins[kSieveCopies][kNB + 4];    // (all of e's exponents: the row's exact total is counted here, too)
    alignas(16) uint64_t lev[3][128];
    alignas(16) uint32_t step[NT / 128][kSieveSteps];    // copies, for lanes that add to one address
    LdsFew   few;
    uint64_t list[kSieveList], small[kWave];             // bits of e << 32 | index
    uint64_t blo[NT], bhi[NT];                           // kept weights by bucket of the token index, halves summed apart
    M96      mass[16];
    struct { M96 D, P, r, err, shift, slack; Edge f; uint64_t w_tie; uint32_t found; } one;  // what one wave worked out for all
    uint64_t sum[16];
    uint64_t rand64;
    uint32_t flag[16];
    uint32_t n, few_n, thr, bucket, unsure;
};

// Is a token that was picked with D, and with P = ceil(top_p * D), the one that the exact D picks?  Both may be off by less than `err` (0: they are
// exact).  As P grows, no token's weight falls -- one above the threshold has its own, one at it a share of what is left, one below none -- and the kept
// mass S grows by what P does, up to what the tie weight's division leaves: so a running sum and the target r, u of S, shift against each other by no
// more than that, whichever thresholds lie in between, and the token is the same if r is further than that from both ends of its place.
// With top_p = 1 P is the row's total, and that is at least the mass of the tokens that have been seen: they are above no such P, however little the rest
// of the row weighs.
__device__ __forceinline__ bool wants_all(const Params &p) { return __float_as_uint(p.top_p) == 0x3F800000u; }        // (of its bits: on scalars)
__device__ __forceinline__ M96 larger_of(const M96 a, const M96 b)
{
    const bool m = a >= b;                               // (by its parts: a choice between two objects would be one between addresses)
    return M96{m ? a.lo : b.lo, m ? a.hi : b.hi};
}
__device__ __forceinline__ bool is_zero(const M96 a) { return !(a.lo | a.hi); }
__device__ __forceinline__ M96 less_by(const M96 a, const M96 b) { return a >= b ? a - b : M96{0ull, 0u}; }
// Is another threshold possible, P being `least` at least and `most` at most: are the tokens above this one enough, or those down to it not?  Then tokens of
// no weight may have some.
__device__ __forceinline__ bool other_threshold(const M96 err, const M96 least, const M96 most, const uint32_t top_k, const uint32_t n_gt, const uint32_t n_eq,
                                                const M96 above, const M96 down)
{
    return !is_zero(err) && ((n_gt && !(above < least)) || (n_gt + n_eq < top_k && !(down >= most)));
}
// How far r and the running sums may shift against each other, P being off by less than err.  The tie weight is (P - above) / n_eq unless that is more than
// it can be, the threshold's own or the share that top_k leaves of it: then S and r do not move.  The divisions leave less than a unit for each of the
// ties, of one threshold or, if another is possible, of two of up to 2^20 tokens.
__device__ __forceinline__ M96 shift_of(const M96 err, const bool other, const M96 least, const uint32_t n_eq, const M96 above, const M96 down, const uint32_t thr,
                                        const uint64_t w_tie)
{
    if (is_zero(err)) return err;
    if (other) return err + M96{(1ull << 21) + 2ull, 0u};
    const M96 n{(uint64_t)n_eq, 0u};
    if (least >= above + m96((u128)w_tie * n_eq) + n || (w_tie == w_of_bits(thr) && least >= down)) return M96{0ull, 0u};
    return err + n + M96{2ull, 0u};
}
// ... of the token whose weight lies at (before, upto] in the running sum
__device__ __forceinline__ bool pick_is_sure(const M96 shift, const M96 before, const M96 upto, const M96 r)
{
    return is_zero(shift) || (before + shift < r && upto >= r + shift);
}

// The level-1 bins of one wave's scan, an octave a lane, from their copies.
template <typename L>
__device__ __forceinline__ void sieve_octaves(OctScan &sc, L &l, const int lane)
{
    sc.load(lane, [&](uint32_t o, uint64_t (&w)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = 0ull;
#pragma unroll
        for (int c = 0; c < kSieveCopies; ++c) {
            const ulonglong2 *two = reinterpret_cast<const ulonglong2 *>(&l.bins[c][o * 4u]);
            const ulonglong2 a = two[0], q = two[1];
            w[0] += a.x; w[1] += a.y; w[2] += q.x; w[3] += q.y;
        }
    });
}

// fn(group of four, bits of their e) over the row, from the logits (x by the definition, sampling.cu:553), eight loads in flight per thread, or four of 1024 threads.
template <int NT, typename F>
__device__ __forceinline__ void sieve_row_pass(const Params &p, const uint32_t row, const float M, F fn)
{
    const uint32_t V4 = (uint32_t)p.V >> 2;
    const char *lrow = logits_row(p, row);
    const bool far = !(__builtin_fabsf(M) <= 100.0f);
    const Frame fr(far ? 0 : (int)M);
    auto e = [&](float x) { return fr.raw(far ? fmaxf(x - M, -1000.0f) : x); };
    const uint4 *pens = p.penalties ? reinterpret_cast<const uint4 *>(p.penalties + (int64_t)row * p.V) : nullptr;
    constexpr int kAhead = NT == kThreads ? 8 : 4;
#pragma unroll 1
    for (uint32_t base = threadIdx.x; base < V4; base += kAhead * NT) {
        uint4 l[kAhead];                                 // (the format is asked once a round: a branch about every load waits for it)
        if (p.dtype == RS_DTYPE_F32) {
#pragma unroll
            for (int u = 0; u < kAhead; ++u) l[u] = reinterpret_cast<const uint4 *>(lrow)[min(base + (uint32_t)(u * NT), V4 - 1u)];
        } else {
            uint2 q[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) q[u] = reinterpret_cast<const uint2 *>(lrow)[min(base + (uint32_t)(u * NT), V4 - 1u)];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                uint32_t w[4];
                widen4(q[u], p.dtype, w);
                l[u] = make_uint4(w[0], w[1], w[2], w[3]);
            }
        }
        if (pens) {
            uint4 q[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) q[u] = pens[min(base + (uint32_t)(u * NT), V4 - 1u)];
            auto less = [&](uint32_t &w, uint32_t pen) { w = __float_as_uint(sf(__uint_as_float(w)) - __uint_as_float(pen)); };
#pragma unroll
            for (int u = 0; u < kAhead; ++u) { less(l[u].x, q[u].x); less(l[u].y, q[u].y); less(l[u].z, q[u].z); less(l[u].w, q[u].w); }
        }
        auto x = [&](uint32_t w) { return sf(__uint_as_float(w) * p.c); };
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
            if (base + (uint32_t)(u * NT) < V4) fn(base + (uint32_t)(u * NT), make_uint4(e(x(l[u].x)), e(x(l[u].y)), e(x(l[u].z)), e(x(l[u].w))));
    }
}

// The row's D from its logits.  `close`: in double precision, 2^-40 of it off at most (D >= 1; a thread adds fewer than 2^13 terms).  Else exactly: all of
// its tokens are counted into L.bins, which is left that way (with e_bits also the e of every token, dead ones as 0).
// The barrier at its start is between the waves that may still read L.bins (each wave searches them for itself in level1) and those that clear them.
template <int NT>
__device__ __forceinline__ M96 sieve_again(const Params &p, LdsSieveFin<NT> &L, const uint32_t row, const float M, const bool close)
{
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    uint4 *eb4 = p.e_bits ? reinterpret_cast<uint4 *>(p.e_bits + (int64_t)row * p.V) : nullptr;
    __syncthreads();
    for (int i = tid; i < kSieveCopies * (kNB + 4); i += NT) (&L.bins[0][0])[i] = 0ull;
    __syncthreads();
    uint64_t *bins = L.bins[lane & (kSieveCopies - 1)];
    double s[2] = {0.0, 0.0};
    sieve_row_pass<NT>(p, row, M, [&](uint32_t i4, const uint4 b) __attribute__((always_inline)) {
        if (close) {
            auto e = [](uint32_t w) { return w < kEMinBits ? 0.0 : (double)__uint_as_float(w); };
            s[0] += e(b.x) + e(b.y); s[1] += e(b.z) + e(b.w);
        } else {
            auto add = [&](uint32_t w) { atomicAdd(reinterpret_cast<unsigned long long *>(&bins[w >> 21]), (unsigned long long)(kPackOne | (w & 0x7FFFFFu))); };
            add(b.x); add(b.y); add(b.z); add(b.w);
            auto live = [](uint32_t w) { return w < kEMinBits ? 0u : w; };
            if (eb4) eb4[i4] = make_uint4(live(b.x), live(b.y), live(b.z), live(b.w));
        }
    });
    if (close) {
        const double mine = wave_sum_f64(s[0] + s[1]);
        if (lane == 0) L.sum[wave] = __builtin_bit_cast(uint64_t, mine);
        __syncthreads();
        double all = 0.0;
        for (int w = 0; w < NT / kWave; ++w) all += __builtin_bit_cast(double, L.sum[w]);
        const uint64_t q = uniform((uint64_t)(all * 0x1p40));
        return M96{q << 23, (uint32_t)(q >> 41)};
    }
    __syncthreads();
    OctScan sc;
    sieve_octaves(sc, L, lane);
    return sc.total();
}

// The old penalties of a row that is read again, from the notes; its waves then all count as having left theirs to the fix-up kernel.  Every wave plays back
// lists of its own, four at a time asked for together: one after the other by the whole workgroup each took two trips to memory.
template <int NT>
__device__ __forceinline__ void sieve_pens_back(const Params &p, const SieveView &v, const uint32_t row)
{
    if (!p.penalties) return;
    constexpr uint32_t W = NT / kWave, kMost = (sieve_pen_cap(8) + kWave - 1u) / kWave;
    const uint32_t lane = threadIdx.x & (kWave - 1u), wave = uniform(threadIdx.x >> 6), lists = v.G * (uint32_t)kWaves;
    rs_u32x4 *pens = reinterpret_cast<rs_u32x4 *>(p.penalties + (int64_t)row * p.V);
    const size_t first = (size_t)row * lists;
    // lane l looks after the wave's l-th list (a finish of W waves has rows of 16 W slices at most)
    const uint32_t its = wave + W * lane;
    const bool have = its < lists;
    uint32_t n = have ? v.noted[first + its] : kSievePenLeft;
    n = n == kSievePenLeft ? 0u : min(n, v.note_cap);
    if (have) v.noted[first + its] = kSievePenLeft;
    for (uint32_t l = 0; l * W < lists; l += 4u) {
        uint32_t at[4][kMost];
        rs_u32x4 old[4][kMost];
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) {
            const size_t rec = (first + min(wave + W * (l + u), lists - 1u)) * v.note_cap;
#pragma unroll
            for (uint32_t k = 0; k < kMost; ++k) {
                const size_t i = rec + min(k * (uint32_t)kWave + lane, v.note_cap - 1u);
                at[u][k] = v.note_at[i]; old[u][k] = reinterpret_cast<const rs_u32x4 *>(v.note_old)[i];
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) {
            const uint32_t of_list = lane_of(n, min(l + u, (uint32_t)kWave - 1u));
#pragma unroll
            for (uint32_t k = 0; k < kMost; ++k)
                if (wave + W * (l + u) < lists && k * (uint32_t)kWave + lane < of_list) pens[at[u][k]] = old[u][k];
        }
    }
    wait_vmem();
    __syncthreads();
}

// NT threads (256 or 512 and a wave that draws the random number, or 1024), PRE units to a wave.
template <int NT> constexpr int sieve_finish_threads() { return NT == 1024 ? NT : NT + kWave; }
//
// What bounds it: the length of its chain, as finish_row's.  The tokens set aside, some hundreds or thousands, are counted in 256 steps of e
// between the bound and the row's largest, and one scan of the counts says down to which step top_k of them lie: these are listed.  A list of
// at most 64 is finished by comparing them with each other; a longer one by level-1 bins with masses, and further digits, of the listed
// tokens alone.  Only when what is listed turns out not to hold the kept set (more tokens in one step than the list takes) are all
// tokens set aside looked at, bins first; and when those do not, the row itself.
template <int NT, int PRE>
__global__ void __launch_bounds__(sieve_finish_threads<NT>()) sieve_finish_kernel(const Params p, const SieveView v)
{
    constexpr int  W = NT / kWave;
    constexpr bool kEach = NT <= 512;                  // every wave works the one-wave steps out for itself
    union LdsAll { LdsSieveFin<NT> f; struct { Lds s; LdsB t; } slow; };
    __shared__ LdsAll u;
    LdsSieveFin<NT> &L = u.f;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = (int)uniform((uint32_t)tid >> 6);
    const uint32_t row = blockIdx.x, G = v.G;

    uint32_t rs[6] = {0u, 0u, 0u, 0u, 0u, 0u};
    uint32_t *rng_st = p.rng + (size_t)row * 16;
    const bool draws = wave == (kEach ? W : W - 1);
    if (draws && !p.inj_u) {
#pragma unroll
        for (int i = 0; i < 6; ++i) rs[i] = rng_st[i];
    }
    auto draw = [&]() __attribute__((always_inline)) {
        if (!p.inj_u) {
            uint32_t o[4];
            philox4x32_10(rs[2], rs[3], rs[4], rs[5], rs[0], rs[1], o);
            if (lane == 0) {
                L.rand64 = ((uint64_t)o[0] << 32) | o[1];
                rng_st[2] = rs[2] + 1u;
                if (rs[2] + 1u == 0u) rng_st[3] = rs[3] + 1u;
            }
        }
    };
    const SieveHdr *hdrs = v.hdr + (size_t)row * G;
    // a slice's mass in units of 2^-40 of the row's frame
    auto mass_in = [&](const uint4 &h, const float M) __attribute__((always_inline)) {
        const float d = M - __builtin_floorf(fkey_inv(h.x));
        const int down = d >= 64.0f ? 64 : (int)d;
        const int sh = (int)(h.w >> 23 & 255u) - 110 - down;    // 2^(ex - 150) in units of 2^-40
        const uint64_t m = (h.w & 0x7FFFFFu) | 0x800000u;
        return sh >= 0 ? m << (sh & 63) : sh > -32 ? m >> (-sh & 63) : 0ull;
    };
    auto is_odd = [&](const uint4 &h, const float M) __attribute__((always_inline)) { return (h.w & kSieveOdd) != 0u && fkey_inv(h.x) >= M - 41.0f; };
    M96 D{0ull, 0u}, P{0ull, 0u}, err{0ull, 0u};
    // D from the slices' sums, and what it may be off by; `dead`: from sums in double precision (bit 1), with tokens that weigh nothing in them (bit 0)
    auto estimate = [&](const uint64_t all, const bool odd, const uint32_t dead) __attribute__((always_inline)) {
        auto part = [&](uint32_t sh) { return M96{(D.lo >> sh) | ((uint64_t)D.hi << (64u - sh)), D.hi >> sh}; };
        D = M96{all << 23, (uint32_t)(all >> 41)};
        if (odd) err = part(kSieveErrOdd);
        else if (dead & 2u) err = part(40u) + M96{1ull << 31, 0u};            // (and 128 slices, cut off at 2^-40)
        else err = part(21u) + part(24u);
        if (odd || dead != 2u) err = err + M96{((uint64_t)p.V << 23) + 2ull, 0u};
        P = ceil_mul(p.top_p, D);
    };
    // ... from its sum in double precision, if there are such; `dead`: with tokens that weigh nothing
    const bool fine = v.fine != nullptr;
    const uint4 *fines = fine ? reinterpret_cast<const uint4 *>(v.fine + (size_t)row * G) : reinterpret_cast<const uint4 *>(hdrs);
    auto fine_in = [&](const uint4 &h, const uint4 &f, const float M, bool &dead) __attribute__((always_inline)) {
        const float d = M - __builtin_floorf(fkey_inv(h.x));
        dead = dead || fkey_inv(f.z) < M - 39.0f;
        return (uint64_t)__builtin_ldexp(__builtin_bit_cast(double, ((uint64_t)f.y << 32) | f.x), 40 - (d >= 64.0f ? 64 : (int)d));
    };
    if (kEach && wave == W) {
        // the wave that draws the random number also adds up the row's mass: neither is wanted before the tokens are listed
        // (bare barriers: what was asked for need not have arrived)
        uint4 h[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) h[k] = *reinterpret_cast<const uint4 *>(&hdrs[min((uint32_t)(lane + k * kWave), G - 1u)]);
        uint4 f[2];                                      // (the headers again where there are no such sums)
#pragma unroll
        for (int k = 0; k < 2; ++k) f[k] = fines[min((uint32_t)(lane + k * kWave), G - 1u)];
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_s_barrier();
        draw();
        const float M = __builtin_floorf(fkey_inv(wave_max_u32(max(h[0].x, h[1].x))));
        uint64_t q = 0;
        bool odd = false, dead = false;
#pragma unroll
        for (int k = 0; k < 2; ++k)
            if ((uint32_t)(lane + k * kWave) < G) {
                q += fine ? fine_in(h[k], f[k], M, dead) : mass_in(h[k], M);
                odd = odd || is_odd(h[k], M);
            }
        estimate(wave_sum(q), __builtin_amdgcn_ballot_w64(odd) != 0ull, (fine ? 2u : 0u) | (__builtin_amdgcn_ballot_w64(dead) != 0ull ? 1u : 0u));
        if (lane == 0) { L.one.D = D; L.one.P = P; L.one.err = err; }
        __syncthreads();
        return;
    }
    // lane i looks after the wave's i-th unit of 64 tokens set aside, unit wave + W i of the row
    const uint32_t sl = (uint32_t)(wave + W * lane) >> (v.units - 1u), half = (uint32_t)(wave + W * lane) & (v.units - 1u), GU = G * v.units;
    const uint64_t *stash = v.stash + (size_t)row * GU * kWave;
    const bool mine = lane < PRE && sl < G;
    constexpr int kHdrs = PRE * W > kWave ? 2 : 1;       // (128 slices at most)
    uint4 keys[kHdrs];
#pragma unroll
    for (int k = 0; k < kHdrs; ++k) keys[k] = *reinterpret_cast<const uint4 *>(&hdrs[min((uint32_t)(lane + k * kWave), G - 1u)]);
    uint4 h = *reinterpret_cast<const uint4 *>(&hdrs[min(sl, G - 1u)]), fh = make_uint4(0u, 0u, 0u, 0u);
    if (!kEach) fh = fines[min(sl, G - 1u)];
    uint64_t pre[PRE];                                   // (units beyond the row's read its last one again)
    auto ask = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PRE; ++i) pre[i] = stash[(size_t)min((uint32_t)(wave + W * i), GU - 1u) * kWave + lane];
    };
    ask();
    auto clear_bins = [&]() __attribute__((always_inline)) {
        for (int c = 0; c < kSieveCopies; ++c)
            for (int i = (int)kBin0 + tid; i < kNB; i += NT) L.bins[c][i] = 0ull;
        for (int i = tid; i < 3 * 128; i += NT) (&L.lev[0][0])[i] = 0ull;
        L.blo[tid] = 0ull; L.bhi[tid] = 0ull;
    };
    for (int i = tid; i < NT / 128 * (int)kSieveSteps; i += NT) (&L.step[0][0])[i] = 0u;
    if (tid == 0) { L.n = 0u; L.few_n = 0u; L.unsure = 0u; }
    // the row's largest token and largest bound, every wave from all headers, behind a bare barrier: what has been asked for need not have arrived
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (!mine) h = make_uint4(0u, 0u, 0u, 0u);
    uint32_t kmax = keys[0].x, kcut = keys[0].z;
#pragma unroll
    for (int k = 1; k < kHdrs; ++k) { kmax = max(kmax, keys[k].x); kcut = max(kcut, keys[k].z); }
    kmax = wave_max_u32(kmax); kcut = wave_max_u32(kcut);
    if (!kEach && draws) draw();
    const float xmax = fkey_inv(kmax);
    const float M = __builtin_floorf(xmax);
    // Complete: every token whose e is larger than that of the largest bound.  (Two values of x may share one e.)
    const uint32_t e_cut = e_bits_of(fkey_inv(max(kcut, 0x00800000u)), M);
    const bool whole = e_cut < kEMinBits;                // ... that is, every live token
    const uint32_t from = max(e_cut + 1u, kEMinBits);
    if constexpr (!kEach) {
        const uint64_t coarse = __builtin_amdgcn_ballot_w64(mine && is_odd(h, M));
        bool dead = false;
        const uint64_t q = wave_sum(mine && half == 0u ? fine ? fine_in(h, fh, M, dead) : mass_in(h, M) : 0ull);
        const uint64_t with_dead = __builtin_amdgcn_ballot_w64(dead);
        if (lane == 0) L.sum[wave] = q | (coarse != 0ull ? 1ull << 63 : 0ull) | (with_dead != 0ull ? 1ull << 62 : 0ull);
    }
    uint32_t b[PRE];                                     // bits of e, 0 for what is not a token of the complete part
    auto look_at = [&](auto each) __attribute__((always_inline)) {
        const bool far = !(__builtin_fabsf(M) <= 100.0f);
        const Frame fr(far ? 0 : (int)M);
        const uint32_t len = max(mine ? h.y & 255u : 0u, half * (uint32_t)kWave) - half * (uint32_t)kWave;     // (of the unit, more than 64 when there is another)
#pragma unroll
        for (int i = 0; i < PRE; ++i) {
            float x = __uint_as_float((uint32_t)(pre[i] >> 32));
            if (far) x = fmaxf(x - M, -1000.0f);
            const uint32_t e = fr.raw(x);
            const bool in = (uint32_t)lane < lane_of(len, (uint32_t)i) && e >= from;
            b[i] = in ? e : 0u;
            if (in) each(e);
        }
    };
    auto to_bins = [&]() __attribute__((always_inline)) {
        const int copy = lane & (kSieveCopies - 1);
        look_at([&](uint32_t e) {
            atomicAdd(reinterpret_cast<unsigned long long *>(&L.bins[copy][e >> 21]), (unsigned long long)(kPackOne | (e & 0x7FFFFFu)));
        });
    };
    const uint32_t top_k = (uint32_t)p.top_k;
    auto total = [&]() __attribute__((always_inline)) {                                 // by then somebody has added up the slices' sums
        if constexpr (kEach) { D = uniform(L.one.D); P = uniform(L.one.P); err = uniform(L.one.err); }
        else {
            uint64_t all = 0, what = 0;
#pragma unroll
            for (int w = 0; w < W; ++w) { all += L.sum[w] & ~(3ull << 62); what |= L.sum[w] >> 62; }
            const uint32_t bits = uniform((uint32_t)what);
            estimate(uniform(all), (bits & 2u) != 0u, (fine ? 2u : 0u) | (bits & 1u));
        }
    };
    // a row finished from a list of at most 64 tokens that holds its kept set: the token + 1 in one lane of the first wave; 0 in `doubts` when
    // nothing is in doubt, 1 when D must be exact, 2 when the list is too short (second wave)
    uint32_t doubts = 0;
    auto from_few = [&](const uint64_t *list, const uint32_t n, const bool all_of_it, const uint32_t rounds) __attribute__((always_inline)) -> uint32_t {
        M96 e = err;
        return few_pick(p, L.few, row, lane, wave, list, n, top_k,
                        [&](const Limbs &upto) __attribute__((always_inline)) {
                            // (see above: more than is listed, whatever that is; without waiting for what it is, which took 0.1 us)
                            if (!all_of_it) return Totals{D, wants_all(p) && n >= top_k && !p.diag ? M96{~0ull, 0x7FFFFFFFu} : P};
                            e = M96{0ull, 0u};           // every live token of the row is there
                            const M96 d = m96(lane_of(upto, 63u));
                            return Totals{d, ceil_mul(p.top_p, d)};
                        }, xmax, &L.rand64, rounds,
                        [&](const M96 &P, bool enough, uint32_t n_gt, uint32_t n_eq, uint32_t thr, const M96 &above, uint64_t w_tie) __attribute__((always_inline)) {
                            const M96 least = less_by(P, e), down = above + m96((u128)w_of_bits(thr) * n_eq);
                            const bool other = other_threshold(e, least, P + e, top_k, n_gt, n_eq, above, down);
                            doubts = !enough ? 2u : 0u;
                            if (lane == 0) L.one.shift = shift_of(e, other, least, n_eq, above, down, thr, w_tie);
                        }, [&](const M96 &slack) __attribute__((always_inline)) { L.one.slack = slack; });
    };
    auto put = [&](uint32_t token, bool few) __attribute__((always_inline)) {
        if (wave <= 1 && doubts) L.unsure = doubts;
        if (token) {
            p.out[row] = (int32_t)(token - 1u);
            if (p.diag) p.diag[row].index = (int32_t)(token - 1u);
        }
        __syncthreads();
        const uint32_t u = uniform(L.unsure);
        return few && u == 0u && !(L.one.slack >= L.one.shift) ? 1u : u;
    };
    // the tokens for which in(i) says so, side by side
    auto list_them = [&](auto in) __attribute__((always_inline)) {
        uint32_t own = 0;
#pragma unroll
        for (int i = 0; i < PRE; ++i) own += in(i) ? 1u : 0u;
        const uint32_t upto = wave_inclusive_scan(own), of_wave = lane63(upto);
        if (of_wave) {
            uint32_t at = 0;
            if (lane == 0) at = atomicAdd(&L.n, of_wave);
            at = uniform(at) + upto - own;
#pragma unroll
            for (int i = 0; i < PRE; ++i)
                if (in(i)) L.list[at++] = ((uint64_t)b[i] << 32) | (uint32_t)pre[i];
        }
    };
    auto tell_policy = [&](const Params &q) {
        if (tid == 0) {
            const uint32_t c = __hip_atomic_fetch_add(&q.hdr->n_need, 1u, __ATOMIC_RELAXED, RS_AGENT);
            if (c == 0u && q.host_words)                 // the call's first such row tells the caller's policy at once
                __hip_atomic_store(q.host_words + q.report, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    };
    // ---- the boundary bin, among the tokens set aside ----
    Edge f{0u, 0u, 0u, 0ull, M96{0ull, 0u}, 0ull};
    M96 goal{0ull, 0u};
    bool found = false;
    auto edge_for_all = [&]() __attribute__((always_inline)) {
        if constexpr (!kEach) {
            if (tid == 0) { L.one.f = f; L.one.D = D; L.one.P = P; L.one.err = err; L.one.found = found ? 1u : 0u; }
            __syncthreads();
            f.at = uniform(L.one.f.at); f.cnt_above = uniform(L.one.f.cnt_above); f.cnt_bin = uniform(L.one.f.cnt_bin);
            f.sum = uniform(L.one.f.sum); f.above = uniform(L.one.f.above); f.bin_sum = uniform(L.one.f.bin_sum);
            D = uniform(L.one.D); P = uniform(L.one.P); err = uniform(L.one.err); found = uniform(L.one.found) != 0u;
        }
    };
    auto level1 = [&](bool known, bool complete) __attribute__((always_inline)) {       // known: D and err are; complete: every live token of the row has been counted
        if (kEach || wave == 0) {
            OctScan sc;
            sieve_octaves(sc, L, lane);
            if (known) P = ceil_mul(p.top_p, D);
            else if (complete) { err = M96{0ull, 0u}; D = sc.total(); P = ceil_mul(p.top_p, D); }
            else total();
            if (wants_all(p)) P = larger_of(sc.total(), P);       // (see wants_all)
            // (the largest that P may be: what is listed then holds the kept set whatever the exact D is, and whether another
            // threshold than this one comes of that is asked behind it)
            goal = P + err;
            found = sc.search(top_k, goal, f);
        }
        edge_for_all();
    };
    // the next digits of the boundary, while more than `most` tokens lie at or above it; tokens(fn): fn(bits of e) for this thread's
    uint32_t lo = 0, span = 0, lv = 2;
    auto digits = [&](uint32_t most, auto tokens) __attribute__((always_inline)) {
#pragma unroll 1
        for (; found && lv <= (uint32_t)kLevels && f.cnt_bin > 1u && f.cnt_above + f.cnt_bin > most; ++lv) {
            const uint32_t dsh = level_shift(lv), exb = lo >> 23;
            uint64_t *hist = L.lev[lv - 2u];
            tokens([&](uint32_t e) {
                if (e - lo <= span) atomicAdd(reinterpret_cast<unsigned long long *>(&hist[(e >> dsh) & 127u]), (unsigned long long)(kPackOne | (e & 0x7FFFFFu)));
            });
            __syncthreads();
            if (kEach || wave == 0) {
                const Edge at = f;
                found = fine_search(lane, [&](int i) { return hist[i]; }, at, top_k, need_of(goal, f.above, exb), f);
            }
            edge_for_all();
            lo |= f.at << dsh;
            span = (1u << dsh) - 1u;
        }
    };
    auto begin = [&]() __attribute__((always_inline)) { lo = f.at << 21; span = (1u << 21) - 1u; lv = 2u; };
    // ---- the steps, and the list ----
    bool again = p.diag != nullptr || p.e_bits != nullptr;               // with the exact D
    bool listed = false;
    uint32_t n_list = 0;
    {
        const uint32_t e_max = e_bits_of(xmax, M);
        const float scale = 255.9f * __builtin_amdgcn_rcpf((float)max(e_max - min(e_max, from), 1u));
        auto step_of = [&](uint32_t e) { return min((uint32_t)((float)(e - from) * scale), kSieveSteps - 1u); };
        look_at([&](uint32_t e) { atomicAdd(&L.step[lane & (NT / 128 - 1)][step_of(e)], 1u); });
        __syncthreads();
        // four steps a lane, the largest first: at which of them top_k tokens are reached, if they fit then
        const uint32_t aim = top_k;
        uint32_t n = 0, step = 0, all = 0;
        if (kEach || wave == 0) {
            uint32_t c[4] = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int k = 0; k < NT / 128; ++k) {
                const uint4 q = reinterpret_cast<const uint4 *>(L.step[k])[63 - lane];
                c[0] += q.w; c[1] += q.z; c[2] += q.y; c[3] += q.x;
            }
            const uint32_t upto = wave_inclusive_scan(c[0] + c[1] + c[2] + c[3]);
            all = lane63(upto);
            n = all;
            if (all > aim) {
                const uint32_t l = (uint32_t)__builtin_ctzll(__builtin_amdgcn_ballot_w64(upto >= aim));
                n = lane_of(upto - c[0] - c[1] - c[2] - c[3], l); step = 256u - 4u * l;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (n < aim) { n += lane_of(c[k], l); step = 255u - 4u * l - (uint32_t)k; }
            }
        }
        if constexpr (!kEach) {
            if (tid == 0) { L.one.f.at = n; L.one.f.cnt_above = step; L.one.f.cnt_bin = all; }
            __syncthreads();
            n = uniform(L.one.f.at); step = uniform(L.one.f.cnt_above); all = uniform(L.one.f.cnt_bin);
        }
        // (fewer than top_k, which are all there are, may still be P)
        listed = n != 0u && n <= kSieveList;
        if (listed) {
            list_them([&](int i) { return b[i] != 0u && step_of(b[i]) >= step; });
            n_list = n;
            if (n > (uint32_t)kWave) clear_bins();
        }
        __syncthreads();
        if (listed && n <= (uint32_t)kWave && !again) {
            total();
            const uint32_t token = from_few(L.list, n, whole && n == all, 0u), in_doubt = put(token, true);
            if (__builtin_expect(in_doubt == 0u, 1)) return;
            again = in_doubt == 1u;
            listed = again;
            __syncthreads();
            if (tid == 0) L.unsure = 0u;
            doubts = 0u;
        }
        if (listed && n > (uint32_t)kWave) {
            for (uint32_t i = (uint32_t)tid; i < n; i += NT) {
                const uint32_t e = (uint32_t)(L.list[i] >> 32);
                atomicAdd(reinterpret_cast<unsigned long long *>(&L.bins[lane & (kSieveCopies - 1)][e >> 21]), (unsigned long long)(kPackOne | (e & 0x7FFFFFu)));
            }
            __syncthreads();
            level1(false, whole && n == all);
            listed = found;
            begin();
        }
    }
    if (__builtin_expect(!listed, 0)) {
        // all tokens set aside, by their bins
        __syncthreads();
        ask();
        clear_bins();
        if (tid == 0) L.n = 0u;
        __syncthreads();
        to_bins();
        __syncthreads();
        level1(false, whole);
        listed = found;
        if (found) {
            begin();
            // a list so long that another kernel is faster (the host's rule): said to the caller's policy
            if (f.cnt_above + f.cnt_bin > min(p.long_list, p.tell_lists ? max(2048u, 3u * top_k) : 0xFFFFFFFFu)) tell_policy(params_again());
            digits(kSieveList, [&](auto fn) {
#pragma unroll
                for (int i = 0; i < PRE; ++i) fn(b[i]);
            });
            n_list = f.cnt_above + f.cnt_bin;
            listed = found && n_list <= kSieveList;
        }
        if (listed) list_them([&](int i) { return b[i] >= lo; });
        __syncthreads();
        if (__builtin_expect(!listed, 0)) {
            // One tie of all the row's tokens (rows of equal logits): every token weighs the tie weight, and the token at which the running sum
            // reaches r follows by division.
            const Params q = params_again();
            const uint64_t rand64 = q.inj_u ? 0ull : L.rand64;
            const bool tie = !mine || ((h.y & kSieveTie) && h.x == kmax);
            const uint64_t not_all = __builtin_amdgcn_ballot_w64(!tie);
            if (lane == 0) L.flag[wave] = not_all != 0ull ? 1u : 0u;
            __syncthreads();
            uint32_t differ = 0;
            for (int w = 0; w < W; ++w) differ |= L.flag[w];
            if (uniform(differ) == 0u) {
                const uint32_t emax = e_bits_of(xmax, M);
                if (q.e_bits)
                    for (uint32_t i = (uint32_t)tid; i < (uint32_t)q.V >> 2; i += NT)
                        reinterpret_cast<uint4 *>(q.e_bits + (int64_t)row * q.V)[i] = make_uint4(emax, emax, emax, emax);
                if (tid == 0) {
                    const u128 all = (u128)w_of_bits(emax) * (uint32_t)q.V;
                    const Target tg = tie_and_target(q, row, rand64, xmax, all, ceil_mul(q.top_p, all), emax, 0u, (uint32_t)q.V, (u128)0, 0u, true);
                    uint32_t lo_i = 0, hi_i = (uint32_t)q.V - 1u;                  // smallest i with (i + 1) * w_tie >= r; r <= V * w_tie
                    while (lo_i < hi_i) {
                        const uint32_t mid = (lo_i + hi_i) >> 1;
                        if ((u128)(mid + 1u) * tg.w_tie >= tg.r) hi_i = mid; else lo_i = mid + 1u;
                    }
                    q.out[row] = (int32_t)lo_i;
                    if (q.diag) q.diag[row].index = (int32_t)lo_i;
                }
                return;
            }
        }
    }
    // ---- threshold and token from the list; a decision too close to call is made again with the row's exact total ----
    bool from_row = false;                               // the list is of the row, not of the tokens set aside
    for (uint32_t sums = 0;; again = true) {             // sums: of the row made so far

        auto from_list = [&](auto fn) {
            for (uint32_t i = (uint32_t)tid; i < n_list; i += NT) fn((uint32_t)(L.list[i] >> 32));
        };
        if (__builtin_expect(again || !listed, 0)) {
            if (sums == 0u) {
                sieve_pens_back<NT>(params_again(), v, row);
                if (tid == 0) __hip_atomic_fetch_add(&params_again().hdr->n_again, 1u, __ATOMIC_RELAXED, RS_AGENT);
            }
            const bool close = sums++ == 0u && listed && !p.diag && !p.e_bits;       // (and exactly when that is not close enough)
            D = sieve_again<NT>(params_again(), L, row, M, close);
            err = close ? M96{(D.lo >> 38) | ((uint64_t)D.hi << 26), 0u} + M96{1ull << 24, 0u} : M96{0ull, 0u};
            if (!listed) {
                // the tokens set aside were not enough, or more than the list holds: the row's own bins, and its tokens at or above the boundary bin
                from_row = true;
                __syncthreads();
                level1(true, false);
                n_list = f.cnt_above + f.cnt_bin;
                if (!found || n_list > kSieveList) break;
                const uint32_t edge = f.at << 21;
                if (tid == 0) L.n = 0u;
                __syncthreads();
                sieve_row_pass<NT>(params_again(), row, M, [&](uint32_t i4, const uint4 e) {
                    auto take = [&](uint32_t w, uint32_t q) {
                        if (w < edge) return;
                        const uint32_t o = atomicAdd(&L.n, 1u);
                        if (o < kSieveList) L.list[o] = ((uint64_t)w << 32) | (i4 * 4u + q);
                    };
                    take(e.x, 0u); take(e.y, 1u); take(e.z, 2u); take(e.w, 3u);
                });
                listed = true;
            }
            __syncthreads();                             // (the bins have been looked at)
            clear_bins();
            if (tid == 0) { L.few_n = 0u; L.unsure = 0u; }
            doubts = 0u;
            __syncthreads();
            from_list([&](uint32_t e) {
                atomicAdd(reinterpret_cast<unsigned long long *>(&L.bins[lane & (kSieveCopies - 1)][e >> 21]), (unsigned long long)(kPackOne | (e & 0x7FFFFFu)));
            });
            __syncthreads();
            level1(true, false);
            begin();
            again = true;
        }
        if (__builtin_expect(found, 1)) digits((uint32_t)kWave, from_list);
        if (__builtin_expect(!found, 0)) {               // (P may be more than is listed)
            if (from_row) break;
            listed = false;
            continue;
        }
        const uint32_t n = f.cnt_above + f.cnt_bin;
        uint32_t token = 0;                              // of the wave that finds it, in one lane: the sampled token + 1
        if (n <= (uint32_t)kWave) {
            // ---- a short list ----
            const uint64_t *list = L.list;
            if (n_list > (uint32_t)kWave) {
                for (uint32_t i = (uint32_t)tid; i < n_list; i += NT) {
                    const uint64_t e = L.list[i];
                    if ((uint32_t)(e >> 32) >= lo) {
                        const uint32_t o = atomicAdd(&L.few_n, 1u);
                        if (o < (uint32_t)kWave) L.small[o] = e;
                    }
                }
                __syncthreads();
                list = L.small;
            }
            token = from_few(list, n_list > (uint32_t)kWave ? n : n_list, false, 0u);
        } else {
            // ---- a longer one ----
            if (span != 0u) {                            // a single token left in the range: the threshold itself
                from_list([&](uint32_t e) { if (e - lo <= span) L.thr = e; });
                __syncthreads();
                lo = uniform(L.thr);
            }
            const uint32_t thr = lo;
            uint64_t w_tie = 0;
            M96 r{0ull, 0u}, shift{0ull, 0u};
            if (kEach || wave == 0) {
                const M96 above = f.above + mass_of(f.sum, thr >> 23);
                const M96 down = above + m96((u128)w_of_bits(thr) * f.cnt_bin);
                M96 least = less_by(P, err);
                if (wants_all(p)) least = larger_of(least, down);
                // (the threshold is that of the largest P: when it need not be the exact one's, so are tie weight and target)
                const bool other = other_threshold(err, least, goal, top_k, f.cnt_above, f.cnt_bin, above, down);
                const Target tg = tie_and_target(p, row, uniform(L.rand64), xmax, wide(D), wide(M96{other ? goal.lo : P.lo, other ? goal.hi : P.hi}), thr, f.cnt_above, f.cnt_bin, wide(above), 0u, tid == 0);
                w_tie = uniform(tg.w_tie); r = uniform(m96(tg.r));
                shift = shift_of(other ? err + err : err, other, least, f.cnt_bin, above, down, thr, w_tie);
            }
            if constexpr (!kEach) {
                if (tid == 0) { L.one.w_tie = w_tie; L.one.r = r; L.one.shift = shift; }
                __syncthreads();
                w_tie = uniform(L.one.w_tie); r = uniform(L.one.r); shift = uniform(L.one.shift);
            }
            // the pick: kept weights by bucket of the token index, NT buckets a step, then the bucket's tokens
            auto weight = [=](uint32_t e) -> uint64_t { return e > thr ? w_of_bits(e) : e == thr ? w_tie : 0ull; };
            constexpr uint32_t kLogNT = NT == 256 ? 8u : NT == 512 ? 9u : 10u;
            uint32_t sh = 32u - (uint32_t)__builtin_clz((uint32_t)p.V - 1u | 1u);
            sh = sh > kLogNT ? sh - kLogNT : 0u;
            uint32_t lo_idx = 0, len = (uint32_t)p.V;
            for (;;) {
                for (uint32_t i = (uint32_t)tid; i < n_list; i += NT) {
                    const uint64_t e = L.list[i];
                    const uint32_t off = (uint32_t)e - lo_idx;
                    if ((uint32_t)(e >> 32) >= thr && off < len) {
                        const uint64_t w = weight((uint32_t)(e >> 32));
                        atomicAdd(reinterpret_cast<unsigned long long *>(&L.blo[off >> sh]), (unsigned long long)(w & 0xFFFFFFFFull));
                        atomicAdd(reinterpret_cast<unsigned long long *>(&L.bhi[off >> sh]), (unsigned long long)(w >> 32));
                    }
                }
                __syncthreads();
                const M96 own = m96((u128)L.blo[tid] + ((u128)L.bhi[tid] << 32));
                L.blo[tid] = 0ull; L.bhi[tid] = 0ull;
                if (tid == 0) L.few_n = 0u;
                M96 inc = m96(wave_inclusive_scan(limbs(own)));
                if (lane == kWave - 1) L.mass[wave] = inc;
                __syncthreads();
                {
                    const Limbs tot = wave_inclusive_scan(limbs(lane < W ? L.mass[lane] : M96{0ull, 0u}));
                    if (wave) inc = inc + m96(lane_of(tot, (uint32_t)wave - 1u));
                }
                const M96 exc = inc - own;
                if (exc < r && inc >= r) { L.bucket = (uint32_t)tid; L.one.r = r - exc; }
                __syncthreads();
                lo_idx += uniform(L.bucket) << sh; len = 1u << sh;
                r = uniform(L.one.r);
                for (uint32_t i = (uint32_t)tid; i < n_list; i += NT) {
                    const uint64_t e = L.list[i];
                    if ((uint32_t)(e >> 32) >= thr && (uint32_t)e - lo_idx < len) {
                        const uint32_t o = atomicAdd(&L.few_n, 1u);
                        if (o < (uint32_t)kWave) L.small[o] = e;
                    }
                }
                __syncthreads();
                const uint32_t ns = uniform(L.few_n);
                if (ns <= (uint32_t)kWave) {
                    if (wave == 0) {
                        const uint64_t e = L.small[min((uint32_t)lane, ns - 1u)];
                        uint32_t rank = 0;
#pragma unroll 4
                        for (uint32_t j = 0; j < ns; ++j) rank += (uint32_t)L.small[j] < (uint32_t)e ? 1u : 0u;
                        if ((uint32_t)lane < ns) { L.few.w[rank] = weight((uint32_t)(e >> 32)); L.few.idx[rank] = (uint32_t)e; }
                        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                        const Limbs one = limbs(M96{(uint32_t)lane < ns ? L.few.w[lane] : 0ull, 0u}), run = wave_inclusive_scan(one);
                        const M96 up = m96(run), bef = m96(run - one);
                        if ((uint32_t)lane < ns && bef < r && up >= r) {
                            token = L.few.idx[lane] + 1u;
                            if (!pick_is_sure(shift, bef, up, r)) doubts = 1u;
                        }
                    }
                    break;
                }
                sh = sh > kLogNT ? sh - kLogNT : 0u;
                __syncthreads();
            }
        }
        const uint32_t in_doubt = put(token, n <= (uint32_t)kWave);
        if (__builtin_expect(in_doubt == 0u, 1)) {
            if (from_row) tell_policy(params_again());
            return;
        }
        if (in_doubt != 1u || !(err.lo | err.hi)) {      // a list that is too short after all
            if (from_row) break;
            listed = false;
        }
    }
    // Thousands of tokens in the boundary bin: the slow way.
    {
        const Params q = params_again();
        const uint64_t rand64 = q.inj_u ? 0ull : L.rand64;
        __syncthreads();                                 // (the row has been summed again: its penalties are back)
        if (NT > kThreads && tid >= kThreads) return;
        __syncthreads();                                 // the LDS is given over
        finish_row_slow(q, u.slow.s, u.slow.t, row, xmax, rand64);
        tell_policy(q);
    }
}

}  // namespace rs
