// 96-bit masses (a row's total weight stays below 2^84) and the scan of a histogram by one wave.
#pragma once

#include "rs_common.h"

namespace rs {

// The mass of a sum of weights in units of the exponent ex (87 <= ex <= 127): 44 bits shifted by up to 40.
__device__ __forceinline__ M96 mass_of(uint64_t sum, uint32_t ex)
{
    const uint32_t sh = ex - 87u;
    return M96{sum << sh, (uint32_t)((sum >> 24) >> (40u - sh))};
}
// The same of a packed bin whose tokens share the exponent ex.
__device__ __forceinline__ M96 pack_m96(uint64_t w, uint32_t ex) { return mass_of((w & kPackMask) + ((w >> 43) << 23), ex); }

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

// What is left to a bin's tokens of one exponent: the mass that must be reached, `above` of which there is already, in units of
// the exponent's weights (2^(ex - 87)), rounded up; all ones when it is out of their reach.
__device__ __forceinline__ uint64_t need_of(M96 P, M96 above, uint32_t ex)
{
    const uint32_t sh = ex - 87u;
    const M96 left = (P - above) + M96{(1ull << sh) - 1ull, 0u};
    return (uint64_t)left.hi >> sh ? ~0ull : (left.lo >> sh) | (((uint64_t)left.hi << 1) << (63u - sh));
}
// Where a scan in order of falling e stopped: the first place at which there are top_k tokens or the mass P, what lies before
// it and what is there (wave-uniform).
struct Edge {
    uint32_t at, cnt_above, cnt_bin;
    uint64_t sum;                                        // of the levels below the first: mass before it since the first level's place, in units of the exponent
    M96      above;                                      // of the first level: mass before it
    uint64_t bin_sum;                                    // of the first level: mass there, in units of the exponent
};

// The 164 bins of level 1 looked at by one wave, an octave of four bins a lane, largest e first: the bins of a lane share
// their exponent, so the lane shifts one sum, a scan over 41 lanes finds the octave, and the bin in it is found on scalars.
struct OctScan {
    uint32_t c[4], cs, before;                           // tokens of the lane's bins, of the lane, of the lanes before
    uint64_t s[4];                                       // the bins' masses in units of the octave's exponent
    Limbs    own, upto;                                  // the lane's mass; with the lanes before
    // octave(o, w): the packed words of octave o (87 to 127), w[0] its smallest bin
    template <typename F>
    __device__ __forceinline__ void load(const int lane, F octave)
    {
        const uint32_t o = (uint32_t)max(127 - lane, 87);
        uint64_t w[4], ss = 0;
        octave(o, w);
        cs = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint64_t q = lane <= 40 ? w[3 - i] : 0ull;
            c[i] = pack_count(q);
            s[i] = (q & kPackMask) + ((uint64_t)c[i] << 23);
            cs += c[i]; ss += s[i];
        }
        own = limbs(mass_of(ss, o));
        before = wave_inclusive_scan(cs) - cs;
        upto = wave_inclusive_scan(own);
    }
    __device__ __forceinline__ M96 total() const { return m96(lane_of(upto, 63u)); }
    // The first bin at which there are top_k tokens or P > 0; false when there is none.
    __device__ __forceinline__ bool search(uint32_t top_k, M96 P, Edge &e) const
    {
        const uint64_t vote = __builtin_amdgcn_ballot_w64(before + cs >= top_k || m96(upto) >= P);
        if (vote == 0ull) return false;
        const uint32_t l = (uint32_t)__builtin_ctzll(vote), ex = 127u - l;
        const M96 mb = m96(lane_of(upto - own, l));
        const uint64_t need = need_of(P, mb, ex);
        e.cnt_above = lane_of(before, l); e.cnt_bin = lane_of(c[0], l);
        uint64_t here = lane_of(s[0], l), sum = 0;
        uint32_t k = 0;
#pragma unroll
        for (uint32_t i = 0; i < 3u; ++i)
            if (k == i && e.cnt_above + e.cnt_bin < top_k && sum + here < need) {
                e.cnt_above += e.cnt_bin; sum += here;
                e.cnt_bin = lane_of(c[i + 1], l); here = lane_of(s[i + 1], l);
                k = i + 1u;
            }
        e.at = ex * 4u + 3u - k;
        e.sum = 0; e.bin_sum = here;
        e.above = mb + mass_of(sum, ex);
        return true;
    }
};

// The next seven bits of one bin's tokens, 128 bins two a lane: `word(i)` bin i, `from` the edge found so far, `need` what
// need_of says of the first level's.  All tokens share the exponent, so masses are 64-bit sums, scanned as two limbs.
template <typename F>
__device__ __forceinline__ bool fine_search(const int lane, F word, const Edge &from, uint32_t top_k, uint64_t need, Edge &e)
{
    const uint64_t w0 = word(127 - 2 * lane), w1 = word(126 - 2 * lane);
    const uint32_t c0 = pack_count(w0), c1 = pack_count(w1), cs = c0 + c1;
    const uint64_t s0 = (w0 & kPackMask) + ((uint64_t)c0 << 23), s1 = (w1 & kPackMask) + ((uint64_t)c1 << 23), ss = s0 + s1;
    const uint32_t ci = wave_inclusive_scan(cs) + from.cnt_above;
    const uint32_t lo = wave_inclusive_scan((uint32_t)ss & 0xFFFFFFu), hi = wave_inclusive_scan((uint32_t)(ss >> 24));
    const uint64_t si = ((uint64_t)hi << 24) + lo + from.sum;
    const uint64_t vote = __builtin_amdgcn_ballot_w64(ci >= top_k || si >= need);
    if (vote == 0ull) return false;
    const uint32_t l = (uint32_t)__builtin_ctzll(vote);
    const bool first = (__builtin_amdgcn_ballot_w64(ci - c1 >= top_k || si - s1 >= need) >> l & 1ull) != 0ull;
    e.at = 127u - 2u * l - (first ? 0u : 1u);
    e.cnt_above = lane_of(ci - cs, l) + (first ? 0u : lane_of(c0, l));
    e.cnt_bin = first ? lane_of(c0, l) : lane_of(c1, l);
    e.sum = lane_of(si - ss, l) + (first ? 0ull : lane_of(s0, l));
    return true;
}

// Scan the level-1 histogram s.g (the first wave; the others wait) for the first bin, largest e first, at which
// (count so far >= top_k) or (mass so far >= P).  The total mass of the histogram is the row total D, and P = ceil(top_p * D)
// is derived from it here.  With LOCAL this workgroup's own histogram s.hm is scanned along and its mass above the
// boundary bin returned in local_above.
template <bool LOCAL, typename L = Lds>
__device__ __forceinline__ Found hist_find_level1(L &s, uint64_t top_k, float top_p, int lane, int wave)
{
    if (wave == 0) {
        auto bins = [](const uint64_t *h) {
            return [h](uint32_t o, uint64_t (&w)[4]) {
#pragma unroll
                for (int i = 0; i < 4; ++i) w[i] = h[o * 4u + (uint32_t)i];
            };
        };
        OctScan sc, own;
        sc.load(lane, bins(s.g));
        if constexpr (LOCAL) own.load(lane, bins(s.hm));
        const M96 D = sc.total(), P = ceil_mul(top_p, D);
        if (lane == 0) { s.D = wide(D); s.P = wide(P); }
        Edge e{0u, 0u, 0u, 0ull, M96{0ull, 0u}, 0ull};
        const bool found = sc.search((uint32_t)min(top_k, (uint64_t)0xFFFFFFFFull), P, e);
        M96 mine{0ull, 0u};
        if constexpr (LOCAL) {
            const uint32_t ex = e.at >> 2, l = 127u - ex, k = 3u - (e.at & 3u);
            if (found) {
                uint64_t part = 0;
#pragma unroll
                for (uint32_t i = 0; i < 3u; ++i)
                    if (i < k) part += lane_of(own.s[i], l);
                mine = m96(lane_of(own.upto - own.own, l)) + mass_of(part, ex);
            }
        }
        if (lane == 0) {
            s.found.bin = found ? e.at : 0u;
            s.found.cnt_above = e.cnt_above; s.found.cnt_bin = e.cnt_bin;
            s.found.mass_above = wide(e.above);
            s.found.local_above = wide(mine);
        }
    }
    __syncthreads();
    return s.found;
}

// The same for a 128-bin level (all tokens share the exponent ex).
template <typename L = Lds>
__device__ __forceinline__ Found hist_find128(L &s, const uint64_t *arr, uint32_t cnt0, u128 mass0, uint64_t top_k, uint32_t ex, int lane, int wave)
{
    if (wave == 0) {
        const M96 above = m96(mass0);
        const Edge from{0u, uniform(cnt0), 0u, 0ull, above, 0ull};
        Edge e = from;
        if (fine_search(lane, [&](int i) { return arr[i]; }, from, (uint32_t)min(top_k, (uint64_t)0xFFFFFFFFull), need_of(uniform(m96((u128)s.P)), uniform(above), ex), e) &&
            lane == 0) {
            s.found.bin = e.at;
            s.found.cnt_above = e.cnt_above; s.found.cnt_bin = e.cnt_bin;
            s.found.mass_above = wide(above + mass_of(e.sum, ex));
        }
    }
    __syncthreads();
    return s.found;
}

// tie_and_target by one wave on values that are the same for all its lanes: on scalars (one thread's 64- and 96-bit
// multiplications and carries go through the vector unit one dependent instruction after the other).
__device__ __forceinline__ Target target_of_wave(const Params &p, uint32_t row, uint64_t rand64, float xmax, u128 D, u128 P, uint32_t thr, uint32_t n_gt,
                                                 uint32_t n_eq, u128 Gm, uint32_t levels, bool write_diag)
{
    return tie_and_target(p, row, uniform(rand64), xmax, wide(uniform(m96(D))), wide(uniform(m96(P))), uniform(thr), uniform(n_gt), uniform(n_eq),
                          wide(uniform(m96(Gm))), levels, write_diag);
}

// ---- a row finished from a list of at most 64 tokens that holds its kept set and its threshold's ties ----
struct LdsFew {
    uint64_t sorted[kWave], w[kWave];
    uint32_t part[4][kWave], idx[kWave];
};
// list: bits of e << 32 | index, in any order, n > 0 of them, with nothing larger left out.  Called by the first four waves
// of the workgroup together (more may call; all meet at its barrier); one wave does it alone when there are few tokens.  Each token is
// compared with every other: its place by falling e, where one scan finds the threshold, and its place by index, where
// another finds the sampled token.  Returns that token + 1 in one lane of wave 0, 0 elsewhere.
// D and P are those of `totals(mass of the whole list)`.  Unless they are LooksAtNothing, `decided` and `picked` are told the outcome: decided() by the second wave,
// which works it out for itself while the first goes on to the token -- the call's P, whether the list is enough, tokens above the threshold and at
// it, the threshold, the mass above it, the tie weight -- and picked() in the sampled token's lane, by how much the target may move either way
// against the running sum.
struct Totals { M96 D, P; };
struct LooksAtNothing {};
template <typename T, typename F = LooksAtNothing, typename K = LooksAtNothing>
__device__ __forceinline__ uint32_t few_pick(const Params &p, LdsFew &s, const uint32_t row, const int lane, const int wave, const uint64_t *list,
                                             const uint32_t n, const uint32_t top_k, T totals, const float xmax,
                                             const uint64_t *rand64, const uint32_t rounds, F decided = F(), K picked = K())
{
    constexpr bool kLook = !std::is_same<F, LooksAtNothing>::value;
    const uint64_t e = list[min((uint32_t)lane, n - 1u)];
    const bool split = n > 16u, in = (uint32_t)lane < n;
    uint32_t larger = 0, before = 0;
    if (wave < (split ? 4 : kLook ? 2 : 1)) {
        const uint32_t each = split ? (n + 3u) >> 2 : n, j0 = kLook && !split ? 0u : (uint32_t)wave * each, j1 = min(n, j0 + each);
#pragma unroll 4
        for (uint32_t j = j0; j < j1; ++j) {
            const uint64_t o = list[j];
            larger += o > e ? 1u : 0u;                   // (equal e: the larger index first)
            before += (uint32_t)o < (uint32_t)e ? 1u : 0u;
        }
        if (split) s.part[wave][lane] = larger | before << 16;
    }
    if (split) __syncthreads();
    if (wave > (kLook ? 1 : 0)) return 0u;
    if (split) {
        const uint32_t c = s.part[0][lane] + s.part[1][lane] + s.part[2][lane] + s.part[3][lane];
        larger = c & 0xFFFFu; before = c >> 16;
    }
    if (in) s.sorted[larger] = e;                        // (two waves: the same words)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const uint32_t b = in ? (uint32_t)(s.sorted[lane] >> 32) : 0u;
    const Limbs own = limbs(M96{in ? w_of_bits(b) : 0ull, 0u}), upto = wave_inclusive_scan(own);
    const uint64_t random = *rand64;                     // (asked for here, wanted for the target)
    const Totals t = totals(upto);
    const M96 D = t.D, P = t.P;
    const uint64_t enough = __builtin_amdgcn_ballot_w64(in && ((uint32_t)lane + 1u >= top_k || m96(upto) >= P));
    const uint32_t thr = lane_of(b, enough ? (uint32_t)__builtin_ctzll(enough) : n - 1u);
    const uint32_t n_gt = (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(b > thr));
    const uint32_t n_eq = (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(b == thr));
    const M96 above = m96(lane_of(upto - own, n_gt));
    const Target tg = tie_and_target(p, row, uniform(random), xmax, wide(D), wide(P), thr, n_gt, n_eq, wide(above), rounds, lane == 0 && (!kLook || wave == 0));
    if constexpr (kLook) {
        if (wave != 0) { decided(P, enough != 0ull, n_gt, n_eq, thr, above, tg.w_tie); return 0u; }
    }
    const M96 r = m96(tg.r);
    if (in) {
        const uint32_t be = (uint32_t)(e >> 32);
        s.w[before] = be > thr ? w_of_bits(be) : be == thr ? tg.w_tie : 0ull;
        s.idx[before] = (uint32_t)e;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const Limbs mine = limbs(M96{in ? s.w[lane] : 0ull, 0u}), run = wave_inclusive_scan(mine);
    const M96 bef = m96(run - mine), with = m96(run);
    const bool is_it = in && bef < r && with >= r;
    if constexpr (kLook) {
        if (is_it) {
            const M96 less = r - bef - M96{1ull, 0u}, more = with - r;
            const bool m = more >= less;
            picked(M96{m ? less.lo : more.lo, m ? less.hi : more.hi});
        }
    }
    return is_it ? s.idx[lane] + 1u : 0u;
}

}  // namespace rs
