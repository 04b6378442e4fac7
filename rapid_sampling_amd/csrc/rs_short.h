// The short-row kernel: one workgroup per row of up to 16384 tokens, the row in its registers, one launch, no waits; any
// kept set, with or without penalties.
//
// What bounds it: the length of its chain.  A row of a few KB arrives in one trip to memory, and what follows is some
// hundred dependent instructions of one or two waves per SIMD between barriers, at four to five cycles each.  So the chain is kept
// short: three barriers and one more for lists of more than 16 tokens; up to eight waves work the one-wave steps out each for
// itself; the random number and the routing report are a wave's of their own; the level-1 bins are looked at an octave a lane
// (OctScan); a kept set of up to 64 tokens, what ties or shares its last digits included, is resolved and picked from by
// comparing all pairs (few_pick), longer ones from the registers; penalties are rewritten as soon as they are read,
// decayed, and only the sampled token's is written again once it is known.
// Measured, us a call, before (general kernel, streaming path or row kernel) -> here: 16 rows of 256, top_k 40 9.15 -> 5.0; 1 of 4096
// 12.0 -> 5.6, with penalties 13.2 -> 5.9; 1024 of 256 28.3 -> 7.0; 64 of 8192 with a nucleus of thousands 13.1 -> 10.8; 256 of 16384, top_k
// 40 12.6 -> 8.6, with penalties 17.6 -> 13.6.
#pragma once

#include "rs_common.h"
#include "rs_mass.h"

namespace rs {

constexpr uint32_t kShortRounds = 10u;                   // rs_row_diag::rounds of a row finished here (as in the row kernel: by one workgroup, from its registers)

template <int W, int R>
struct LdsShort {
    static constexpr uint32_t kCopies = W * R >= 64 ? 8u : 4u;      // of each level-1 bin while it is counted (lane l adds to copy l mod that)
    static constexpr uint32_t kPlane  = kNB + 4u;        // words from copy to copy: the copies of a bin lie in different banks, an octave's bins together
    alignas(16) uint64_t hr[kCopies * kPlane];
    alignas(16) uint64_t lev[3][128];                    // levels 2 to 4
    LdsFew   few;
    uint64_t list[kWave];
    M96      mass[W];
    struct { M96 D, P, r; Edge f; uint64_t w_tie; } one; // what one wave worked out for all (sixteen waves)
    uint64_t rand64;
    uint32_t wmax[W], n, thr, token;
};

// Wave w of W holds the stretch of ceil(V / 4 / W) groups of four tokens from group w * that on, lane l its groups j * 64 + l
// (j < R): index order is wave, then j, then lane, then token.  Up to two waves per SIMD work the one-wave steps out each
// for itself and leave the random number to a wave of its own; of sixteen the first does them for all and the last draws.
template <int W> constexpr int short_threads() { return (W <= 8 ? W + 1 : W) * kWave; }
// Waves a SIMD must hold: two workgroups of sixteen waves share a compute unit in 64 registers.  The four groups of a thread took 66
// when left alone, one workgroup a compute unit: 512 rows of 16384, top_k 40 16.9 us a call, in 64 13.5; 384 with a top_k of 300 25.2
// and 20.6 (with penalties 88 are needed, which no bound brings down to 64).
template <bool PEN, int W, int R> constexpr int short_waves() { return W == 16 && !PEN ? 8 : 1; }
template <int DT, bool PEN, int W, int R>
__global__ void __launch_bounds__(short_threads<W>(), (short_waves<PEN, W, R>())) short_kernel(const Params p)
{
    constexpr bool kEach = W <= 8;
    constexpr uint32_t kCopies = LdsShort<W, R>::kCopies, kPlane = LdsShort<W, R>::kPlane;
    __shared__ LdsShort<W, R> L;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = (int)uniform((uint32_t)tid >> 6);
    const uint32_t row = blockIdx.x;
    // the row's random number, and the report on the streaming call before this one (report_begin)
    const bool draws = wave == (kEach ? W : W - 1), reporter = draws && row == 0u && lane == 0 && p.host_words != nullptr;
    PrevCall prev;
    prev.slow_rows = 0; prev.meta = 0;
    uint32_t *st = p.rng + (size_t)row * 16;
    uint32_t rs[6] = {0u, 0u, 0u, 0u, 0u, 0u};
    if (draws && !p.inj_u) {
#pragma unroll
        for (int i = 0; i < 6; ++i) rs[i] = st[i];
    }
    if (reporter) prev = report_begin(p);
    auto draw = [&]() {
        if (!p.inj_u) {
            uint32_t o[4];
            philox4x32_10(rs[2], rs[3], rs[4], rs[5], rs[0], rs[1], o);
            if (lane == 0) {
                L.rand64 = ((uint64_t)o[0] << 32) | o[1];
                st[2] = rs[2] + 1u;
                if (rs[2] + 1u == 0u) st[3] = rs[3] + 1u;
            }
        }
        if (reporter) report_end(p, prev, false);
    };
    if (kEach && wave == W) {
        __builtin_amdgcn_s_barrier();                    // (bare: what was asked for above need not have arrived)
        __builtin_amdgcn_s_barrier();
        draw();
        __syncthreads();
        return;
    }
    const uint32_t V4 = (uint32_t)p.V >> 2, per = (V4 + (uint32_t)W - 1u) / (uint32_t)W;
    const uint32_t g0 = (uint32_t)wave * per + (uint32_t)lane;             // this thread's first group
    const uint32_t g_end = min(((uint32_t)wave + 1u) * per, V4);           // end of the wave's stretch
    const char *lrow = logits_row(p, row);
    float4 *pn4 = PEN ? reinterpret_cast<float4 *>(p.penalties + (int64_t)row * p.V) : nullptr;
    auto group = [&](int j) { return g0 + (uint32_t)(j * kWave); };

    // slots past the end of the stretch read the row's last group again (harmless for the maximum and the probe) and
    // are set aside before anything is counted
    uint32_t eb[R * 4];                                  // l, then x, then bits(e)
    float4 pen[PEN ? R : 1];
    if constexpr (DT == RS_DTYPE_F32) {
        const uint4 *lg = reinterpret_cast<const uint4 *>(lrow);
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const uint4 l = load_once(lg + min(group(j), V4 - 1u));
            eb[j * 4 + 0] = l.x; eb[j * 4 + 1] = l.y; eb[j * 4 + 2] = l.z; eb[j * 4 + 3] = l.w;
        }
    } else {
        const uint2 *lh = reinterpret_cast<const uint2 *>(lrow);
        uint2 h[R];
#pragma unroll
        for (int j = 0; j < R; ++j) h[j] = load_once(lh + min(group(j), V4 - 1u));
#pragma unroll
        for (int j = 0; j < R; ++j) widen4(h[j], DT, &eb[j * 4]);
    }
    if constexpr (PEN) {
#pragma unroll
        for (int j = 0; j < R; ++j) pen[j] = pn4[min(group(j), V4 - 1u)];
    }
    // (of the level-1 bins only those of live tokens are ever read)
    constexpr uint32_t kLive16 = (uint32_t)(kNB - (int)kBin0) / 2u;        // 16-byte words of one copy's live bins
    for (uint32_t i = (uint32_t)tid; i < kCopies * kLive16; i += W * kWave) {
        const uint32_t c = i / kLive16;
        reinterpret_cast<uint4 *>(L.hr)[(c * kPlane + kBin0) / 2u + (i - c * kLive16)] = make_uint4(0u, 0u, 0u, 0u);
    }
    if (tid < 192) reinterpret_cast<uint4 *>(L.lev)[tid] = make_uint4(0u, 0u, 0u, 0u);
    if (tid == 0) L.n = 0u;

    // x = sf((sf(l) - pen) * c), without the clean-ups unless a NaN or an infinity shows up (see slice_load)
    constexpr int kSpecial = 0x207;
    float probe = 0.0f, lmax = -3.402823466e+38f;
#pragma unroll
    for (int j = 0; j < R; ++j) {
        float x[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float l = __uint_as_float(eb[j * 4 + q]);
            if constexpr (PEN) x[q] = (l - (q == 0 ? pen[j].x : q == 1 ? pen[j].y : q == 2 ? pen[j].z : pen[j].w)) * p.c;
            else x[q] = l * p.c;
            eb[j * 4 + q] = __float_as_uint(x[q]);
        }
        probe = __builtin_fmaf(x[0], x[1], probe);
        probe = __builtin_fmaf(x[2], x[3], probe);
        lmax = fmaxf(fmaxf(lmax, x[0]), fmaxf(x[1], fmaxf(x[2], x[3])));
    }
    if (__builtin_amdgcn_classf(probe, kSpecial)) {
        lmax = -3.402823466e+38f;
#pragma unroll
        for (int j = 0; j < R; ++j) {
            float x[4];
            if constexpr (PEN) {
                const float4 l = load_logits4(lrow, min(group(j), V4 - 1u), DT);
                x[0] = sf((sf(l.x) - pen[j].x) * p.c); x[1] = sf((sf(l.y) - pen[j].y) * p.c);
                x[2] = sf((sf(l.z) - pen[j].z) * p.c); x[3] = sf((sf(l.w) - pen[j].w) * p.c);
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) x[q] = sf(__uint_as_float(eb[j * 4 + q]));
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) { lmax = fmaxf(lmax, x[q]); eb[j * 4 + q] = __float_as_uint(x[q]); }
        }
    }
    {
        const uint32_t k = wave_max_u32(fkey(lmax));
        if (lane == 0) L.wmax[wave] = k;
    }
    __syncthreads();
    uint32_t kmax = L.wmax[0];
#pragma unroll
    for (int w = 1; w < W; ++w) kmax = max(kmax, L.wmax[w]);
    const float xmax = fkey_inv(uniform(kmax));
    const float M = __builtin_floorf(xmax);

    // e (not clamped at 2^-40: what lies below is dead and lands in bins nobody looks at) and level 1
    const Frame fr = frame_of(M, eb);
    const uint32_t copy = ((uint32_t)lane & (kCopies - 1u)) * kPlane;
#pragma unroll
    for (int j = 0; j < R; ++j) {
        if (group(j) < g_end) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t b = fr.raw(__uint_as_float(eb[j * 4 + q]));
                eb[j * 4 + q] = b;
                atomicAdd(reinterpret_cast<unsigned long long *>(&L.hr[(b >> 21) + copy]), (unsigned long long)(kPackOne | (b & 0x7FFFFFu)));
            }
        } else {
            eb[j * 4] = 0; eb[j * 4 + 1] = 0; eb[j * 4 + 2] = 0; eb[j * 4 + 3] = 0;
        }
    }
    if constexpr (PEN) {
        // Every penalty but the sampled token's becomes fma(pen, decay, 0), whatever is sampled: written now, while the rest
        // is worked out.  Groups of four that are all +0.0 stay +0.0 under a finite decay.
        const bool finite = p.decay - p.decay == 0.0f;
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const float4 q = pen[j];
            if (group(j) < g_end &&
                ((__float_as_uint(q.x) | __float_as_uint(q.y) | __float_as_uint(q.z) | __float_as_uint(q.w)) != 0u || !finite))
                pn4[group(j)] = make_float4(__builtin_fmaf(q.x, p.decay, 0.0f), __builtin_fmaf(q.y, p.decay, 0.0f),
                                            __builtin_fmaf(q.z, p.decay, 0.0f), __builtin_fmaf(q.w, p.decay, 0.0f));
        }
    }
    if (__builtin_expect(p.e_bits != nullptr, 0)) {
        // diagnostics: e of every token, dead tokens as 0
        uint4 *dst = reinterpret_cast<uint4 *>(p.e_bits + (int64_t)row * p.V);
        auto live = [](uint32_t b) { return b < kEMinBits ? 0u : b; };
#pragma unroll
        for (int j = 0; j < R; ++j)
            if (group(j) < g_end) dst[group(j)] = make_uint4(live(eb[j * 4]), live(eb[j * 4 + 1]), live(eb[j * 4 + 2]), live(eb[j * 4 + 3]));
    }
    __syncthreads();

    // ---- the boundary bin, with D and P ----
    const uint32_t top_k = (uint32_t)p.top_k;
    M96 D{0ull, 0u}, P{0ull, 0u};
    Edge f{0u, 0u, 0u, 0ull, M96{0ull, 0u}, 0ull};
    // a step of one wave: every wave does it for itself, or the first one's result goes by way of LDS
    auto edge_for_all = [&]() {
        if constexpr (!kEach) {
            if (tid == 0) L.one.f = f;
            __syncthreads();
            f.at = uniform(L.one.f.at); f.cnt_above = uniform(L.one.f.cnt_above); f.cnt_bin = uniform(L.one.f.cnt_bin);
            f.sum = uniform(L.one.f.sum); f.above = uniform(L.one.f.above); f.bin_sum = uniform(L.one.f.bin_sum);
        }
    };
    if (kEach || wave == 0) {
        OctScan sc;
        sc.load(lane, [&](uint32_t o, uint64_t (&w)[4]) {
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = 0ull;
#pragma unroll
            for (uint32_t c = 0; c < kCopies; ++c) {
                const ulonglong2 *two = reinterpret_cast<const ulonglong2 *>(&L.hr[c * kPlane + o * 4u]);
                const ulonglong2 a = two[0], b = two[1];
                w[0] += a.x; w[1] += a.y; w[2] += b.x; w[3] += b.y;
            }
        });
        D = sc.total();
        P = ceil_mul(p.top_p, D);
        sc.search(top_k, P, f);
        if (!kEach && tid == 0) { L.one.D = D; L.one.P = P; }
    }
    if (!kEach && draws) draw();
    edge_for_all();
    if constexpr (!kEach) { D = uniform(L.one.D); P = uniform(L.one.P); }

    // ---- its next digits, while more tokens lie at or above it than a short list holds ----
    const uint32_t ex = f.at >> 2;
    uint32_t lo = f.at << 21, span = (1u << 21) - 1u;
    if (f.cnt_above + f.cnt_bin > (uint32_t)kWave) {
        if (kEach) __syncthreads();                      // (the third of the wave that draws)
        const uint64_t need = need_of(P, f.above, ex);
        if (f.cnt_above == 0u) {
            // a boundary bin that is one tie of the row's largest token: counting it would queue its tokens up at one address
            const uint32_t emax = e_bits_of(xmax, M);
            if (f.bin_sum == (uint64_t)f.cnt_bin * ((emax & 0x7FFFFFu) | 0x800000u)) { lo = emax; span = 0u; }
        }
#pragma unroll 1
        for (uint32_t lv = 2; lv <= (uint32_t)kLevels && f.cnt_bin > 1u && span != 0u && f.cnt_above + f.cnt_bin > (uint32_t)kWave; ++lv) {
            const uint32_t dsh = level_shift(lv);
            uint64_t *hist = L.lev[lv - 2u];
#pragma unroll
            for (int i = 0; i < R * 4; ++i)
            {
                const uint32_t b = opaque(eb[i]);
                if (b - lo <= span) atomicAdd(reinterpret_cast<unsigned long long *>(&hist[(b >> dsh) & 127u]), (unsigned long long)(kPackOne | (b & 0x7FFFFFu)));
            }
            __syncthreads();
            if (kEach || wave == 0) {
                const Edge from = f;
                fine_search(lane, [&](int i) { return hist[i]; }, from, top_k, need, f);
            }
            edge_for_all();
            lo |= f.at << dsh;
            span = (1u << dsh) - 1u;
        }
    }
    const uint32_t n = f.cnt_above + f.cnt_bin;

    uint32_t token = 0;                                  // of the wave that finds it, in one lane: the sampled token + 1
    if (n <= (uint32_t)kWave) {
        // ---- a short list ----
        uint32_t mine = 0;
#pragma unroll
        for (int i = 0; i < R * 4; ++i) mine += eb[i] >= lo ? 1u : 0u;
        const uint32_t upto = wave_inclusive_scan(mine), of_wave = lane63(upto);
        if (of_wave) {
            uint32_t at = 0;
            if (lane == 0) at = atomicAdd(&L.n, of_wave);
            at = uniform(at) + upto - mine;
#pragma unroll
            for (int i = 0; i < R * 4; ++i)
                if (eb[i] >= lo) L.list[at++] = ((uint64_t)eb[i] << 32) | (group(i >> 2) * 4u + (uint32_t)(i & 3));
        }
        __syncthreads();
        token = few_pick(p, L.few, row, lane, wave, L.list, n, top_k, [&](const Limbs &) { return Totals{D, P}; }, xmax, &L.rand64, kShortRounds);
    } else {
        // ---- a longer one: everything from the registers ----
        if (span != 0u) {                                // a single token left in the range: the threshold itself
#pragma unroll
            for (int i = 0; i < R * 4; ++i)
                if (eb[i] - lo <= span) L.thr = eb[i];
            __syncthreads();
            lo = uniform(L.thr);
        }
        const uint32_t thr = lo;
        uint64_t w_tie = 0;
        M96 r{0ull, 0u};
        if (kEach || wave == 0) {
            const Target tg = tie_and_target(p, row, uniform(L.rand64), xmax, wide(D), wide(P), thr, f.cnt_above, f.cnt_bin,
                                             wide(f.above + mass_of(f.sum, ex)), kShortRounds, tid == 0);
            w_tie = uniform(tg.w_tie); r = uniform(m96(tg.r));
        }
        if constexpr (!kEach) {
            if (tid == 0) { L.one.w_tie = w_tie; L.one.r = r; }
            __syncthreads();
            w_tie = uniform(L.one.w_tie); r = uniform(L.one.r);
        }

        // the pick: the kept weights of every wave's stretch, then of the stretch that holds the target, a group a lane
        auto weight = [=](uint32_t b) -> uint64_t { return b > thr ? w_of_bits(b) : b == thr ? w_tie : 0ull; };
        auto of_group = [&](int j) {
            return M96{weight(opaque(eb[j * 4])), 0u} + M96{weight(opaque(eb[j * 4 + 1])), 0u} + M96{weight(opaque(eb[j * 4 + 2])), 0u} +
                   M96{weight(opaque(eb[j * 4 + 3])), 0u};
        };
        M96 sum{0ull, 0u};
#pragma unroll
        for (int j = 0; j < R; ++j) {
            sum = sum + of_group(j);
            // (group by group: or all the weights are worked out first, two registers each, and summed as a tree)
            asm volatile("" : "+v"(sum.lo), "+v"(sum.hi));
        }
        const M96 whole = m96(lane_of(wave_inclusive_scan(limbs(sum)), 63u));
        if (lane == 0) L.mass[wave] = whole;
        __syncthreads();
        const M96 ours = lane < W ? L.mass[lane] : M96{0ull, 0u};
        const Limbs ol = limbs(ours), upto_w = wave_inclusive_scan(ol);
        const uint32_t owner = (uint32_t)__builtin_ctzll(__builtin_amdgcn_ballot_w64(m96(upto_w) >= r));     // 1 <= r <= the sum of all kept weights
        r = r - m96(lane_of(upto_w - ol, owner));
        if ((uint32_t)wave == owner) {
            bool found = false;
#pragma unroll
            for (int j = 0; j < R; ++j) {
                if (found) continue;
                const M96 own = of_group(j);
                const Limbs gl = limbs(own), upto = wave_inclusive_scan(gl);
                const M96 all = m96(lane_of(upto, 63u));
                if (!(all >= r)) { r = r - all; continue; }
                found = true;
                const M96 inc = m96(upto), exc = m96(upto - gl);
                if (exc < r && inc >= r) {               // exactly one lane
                    uint32_t q = 0;
                    M96 run = exc + M96{weight(eb[j * 4]), 0u};
                    if (!(run >= r)) { q = 1; run = run + M96{weight(eb[j * 4 + 1]), 0u}; }
                    if (q == 1u && !(run >= r)) { q = 2; run = run + M96{weight(eb[j * 4 + 2]), 0u}; }
                    if (q == 2u && !(run >= r)) q = 3;
                    token = group(j) * 4u + q + 1u;
                }
            }
        }
    }
    if (token) {
        p.out[row] = (int32_t)(token - 1u);
        if (p.diag) p.diag[row].index = (int32_t)(token - 1u);
        if (PEN) L.token = token - 1u;
    }
    if constexpr (PEN) {
        // the sampled token's penalty, by the thread that wrote its group before (reference: sampling.cu:427-437)
        __syncthreads();
        const uint32_t idx = uniform(L.token);
#pragma unroll
        for (int j = 0; j < R; ++j)
            if (group(j) == idx >> 2 && group(j) < g_end) {
                const uint32_t q = idx & 3u;
                const float old = q == 0u ? pen[j].x : q == 1u ? pen[j].y : q == 2u ? pen[j].z : pen[j].w;
                reinterpret_cast<float *>(pn4)[idx] = __builtin_fmaf(old, p.decay, old == 0.0f ? p.presence : p.repetition);
            }
    }
}

}  // namespace rs
