// The row kernel: one workgroup of 1024 threads per row (512 in calls of many rows of up to 32768 tokens, two
// such workgroups to a compute unit: launch_row), the whole row (up to 65536 tokens) in its
// registers, one launch, one read of the logits, no workspace, no waits, no other kernel.
//
// A row of up to 65536 tokens fits the registers of one compute unit (64 tokens per thread), and
// then everything the other paths exchange between workgroups or kernels stays inside one
// workgroup: the maximum, e, the level-1 histogram in LDS, the radix selection of the threshold
// level by level (level 2 on the registers, the deeper ones on a list of the boundary bin's tokens
// in LDS when they fit), tie weight and target, and the pick by sums and scans of the kept weights
// in index order.  With more than a sixth of the row at or above the boundary bin its time hardly depends on the
// kept set, only on the row: it is the time of the vector instructions of e and of three passes over the
// registers, 64 tokens per thread with four waves per SIMD; with less, everything behind e and level 1 reads lists
// (below), and the call takes a sixth to a fifth less.  Measured with more, launch included: 14-18 us for 8192 tokens,
// 26 for 32768, 33 for 50304, 42 for 65536; a call of B rows takes ceil(B / 256) such times, or ceil(B / 512) times 17, 24 and 39 us in
// rows of 8192, 16384 and 32768 tokens.  For kept sets of thousands of
// tokens in calls of 64 rows and more that is less than the general kernel's exchanges or the wide
// paths' launches cost; small calls and small kept sets are better off elsewhere.  Same integers as
// every other path.
#pragma once

#include "rs_common.h"
#include "rs_mass.h"

namespace rs {

constexpr int      kRowT      = 1024;                    // threads of the row kernel
constexpr int      kRowW      = kRowT / kWave;
constexpr int      kRowR      = 16;                      // groups of four tokens per thread at most: rows of up to 65536 tokens
static_assert(kRowMaxV == kRowT * kRowR * 4, "the row kernel's registers hold kRowMaxV tokens");
constexpr uint32_t kRowListW  = 768u;                    // tokens of the boundary bin a wave can list for levels 3 and 4
constexpr uint32_t kRowList   = kRowListW * 12u;         // the row's boundary bin is listed when it holds no more than this (16 waves: room to spare for uneven shares)
constexpr uint32_t kRowKeptW  = kRowListW / 2u;          // the same lists with 64-bit entries: tokens at or above the boundary bin, with their places
constexpr uint32_t kRowKept   = kRowKeptW * 12u;         // listed when there are no more than this in the row
constexpr uint32_t kRowFew    = 16u;                     // tokens of a boundary that are compared with each other
constexpr uint32_t kRowRounds = 10u;                     // DiagRow::rounds of a row finished here

struct LdsRowS {                      // what the shared helpers work on
    u128     D, P;
    Found    found;
    u128     bc128[2];
    uint64_t g[kNB];                  // the row's level-1 bins
    uint64_t hm[128];                 // a deeper level's bins
    uint64_t bc64[2];
    uint32_t bc32[8];
};
static_assert(kRowW * kRowListW / 2 >= (uint32_t)kNB * 8u, "the lists lie where the copies of the level-1 bins were");
struct LdsRow {
    LdsRowS  s;
    alignas(16) uint64_t hr8[kRowW * kRowListW / 2];   // level 1 while it is counted: eight copies of each bin (the first kNB * 8
                                      // words); later the waves' lists of the boundary bin's tokens (all of it)
    uint64_t lev[128 * 4];            // a deeper level while it is counted: four copies
    u128     wq[kRowW];               // per wave: kept weight of its stretch of the row
    u128     wq4[kRowW][4];           // the same, a quarter of the wave's groups at a time
    uint32_t nolist;                  // a wave's share of the boundary bin did not fit its list
    uint32_t nsmall, small[kRowFew];  // the last few tokens among which the threshold is
    uint32_t nokept;                  // the same for the list of all tokens at or above the boundary bin
    uint32_t wu[kRowW];
    uint64_t rand64;
};

constexpr uint32_t kRowStage = 128u;                     // groups on their way to a wave's list
template <int W> struct LdsRowStage {
    alignas(16) uint4 grp[W][kRowStage];
    uint32_t at[W][kRowStage];
};

template <int W>
__device__ __forceinline__ uint32_t row_max_u32(LdsRow &L, uint32_t v, int lane, int wave)
{
    v = wave_max_u32(v);
    if (lane == 0) L.wu[wave] = v;
    __syncthreads();
    uint32_t r = L.wu[0];
#pragma unroll
    for (int w = 1; w < W; ++w) r = max(r, L.wu[w]);
    return r;
}

// Wave w holds the stretch of G = ceil(V / 4 / 16) groups of four tokens from group w * G on, lane l its
// groups w * G + j * 64 + l (j < R): a load instruction of a wave reads 1 KB in one piece, and index
// order is wave, then j, then lane, then token.
template <int DT, int NT, int R>      // the logits' type; threads, groups per thread (R * NT >= V / 4)
__global__ void __launch_bounds__(NT, 4) row_kernel(const Params p)
{
    constexpr int kRowT = NT, kRowW = NT / kWave, kRowR = R;
    constexpr uint32_t kRowListW = rs::kRowListW * (uint32_t)(rs::kRowW / kRowW), kRowKeptW = rs::kRowKeptW * (uint32_t)(rs::kRowW / kRowW);
    __shared__ LdsRow L;
    __shared__ LdsRowStage<NT / kWave> stage;
    LdsRowS &s = L.s;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    const uint32_t row = blockIdx.x;
    const uint32_t V4 = (uint32_t)p.V >> 2;
    const uint32_t G = (V4 + (uint32_t)kRowW - 1u) / (uint32_t)kRowW;
    const uint32_t g0 = (uint32_t)wave * G + (uint32_t)lane;               // this thread's first group
    const uint32_t g_end = min(((uint32_t)wave + 1u) * G, V4);             // end of the wave's stretch
    const char *lrow = logits_row(p, row);
    // the call's first thread reports on the streaming call before it, if there was one (report_begin)
    const bool reporter = blockIdx.x == 0 && tid == 0 && p.host_words != nullptr;
    PrevCall prev;
    prev.slow_rows = 0; prev.meta = 0;
    if (reporter) prev = report_begin(p);
    for (int i = (int)kBin0 * 4 + tid; i < kNB * 4; i += kRowT) reinterpret_cast<uint4 *>(L.hr8)[i] = make_uint4(0u, 0u, 0u, 0u);       // (the bins of live tokens)
    if (tid < 128 * 4) L.lev[tid] = 0ull;
    if (tid == 0) { L.nolist = 0u; L.nokept = 0u; L.nsmall = 0u; }

    // token (g0 + j * 64) * 4 + q sits in register j * 4 + q; slots past the end of the stretch read the
    // row's last group again (harmless for the maximum and the probe) and are set aside before anything is counted
    uint32_t eb[kRowR * 4];                              // l, then x, then bits(e)
    if constexpr (DT == RS_DTYPE_F32) {
        const uint4 *lg = reinterpret_cast<const uint4 *>(lrow);
#pragma unroll
        for (int j = 0; j < kRowR; ++j) {
            const uint4 l = load_once(lg + min(g0 + (uint32_t)(j * kWave), V4 - 1u));
            eb[j * 4 + 0] = l.x; eb[j * 4 + 1] = l.y; eb[j * 4 + 2] = l.z; eb[j * 4 + 3] = l.w;
        }
    } else {
        const uint2 *lh = reinterpret_cast<const uint2 *>(lrow);
        uint2 h[kRowR];
#pragma unroll
        for (int j = 0; j < kRowR; ++j) h[j] = load_once(lh + min(g0 + (uint32_t)(j * kWave), V4 - 1u));
#pragma unroll
        for (int j = 0; j < kRowR; ++j) widen4(h[j], DT, &eb[j * 4]);
    }
    // the row's random number, drawn while the loads are in flight; the row is always finished here
    if (tid == kWave && !p.inj_u) {
        uint32_t *rng_st = p.rng + (size_t)row * 16;
        uint32_t rs[6], o[4];
#pragma unroll
        for (int i = 0; i < 6; ++i) rs[i] = rng_st[i];
        philox4x32_10(rs[2], rs[3], rs[4], rs[5], rs[0], rs[1], o);
        L.rand64 = ((uint64_t)o[0] << 32) | o[1];
        rng_st[2] = rs[2] + 1u;
        if (rs[2] + 1u == 0u) rng_st[3] = rs[3] + 1u;
    }
    // x = l * c unless a NaN or an infinity shows up (see stream_kernel)
    constexpr int kSpecial = 0x207;
    float probe = 0.0f;
    float lmax = -3.402823466e+38f;
#pragma unroll
    for (int j = 0; j < kRowR; ++j) {
        const float x0 = __uint_as_float(eb[j * 4]) * p.c, x1 = __uint_as_float(eb[j * 4 + 1]) * p.c;
        const float x2 = __uint_as_float(eb[j * 4 + 2]) * p.c, x3 = __uint_as_float(eb[j * 4 + 3]) * p.c;
        probe = __builtin_fmaf(x0, x1, probe);
        probe = __builtin_fmaf(x2, x3, probe);
        lmax = fmaxf(fmaxf(lmax, x0), fmaxf(x1, fmaxf(x2, x3)));
        eb[j * 4 + 0] = __float_as_uint(x0); eb[j * 4 + 1] = __float_as_uint(x1);
        eb[j * 4 + 2] = __float_as_uint(x2); eb[j * 4 + 3] = __float_as_uint(x3);
    }
    if (__builtin_amdgcn_classf(probe, kSpecial)) {
        lmax = -3.402823466e+38f;
#pragma unroll
        for (int j = 0; j < kRowR; ++j) {
            const float x0 = sf(__uint_as_float(eb[j * 4])), x1 = sf(__uint_as_float(eb[j * 4 + 1]));
            const float x2 = sf(__uint_as_float(eb[j * 4 + 2])), x3 = sf(__uint_as_float(eb[j * 4 + 3]));
            lmax = fmaxf(lmax, fmaxf(fmaxf(x0, x1), fmaxf(x2, x3)));
            eb[j * 4 + 0] = __float_as_uint(x0); eb[j * 4 + 1] = __float_as_uint(x1);
            eb[j * 4 + 2] = __float_as_uint(x2); eb[j * 4 + 3] = __float_as_uint(x3);
        }
    }
    if (reporter) report_end(p, prev, false);
    const uint32_t kmax = row_max_u32<kRowW>(L, fkey(lmax), lane, wave);
    const float xmax = fkey_inv(kmax);
    const float M = __builtin_floorf(xmax);

    // e (not clamped at 2^-40: what lies below is dead and lands in bins nobody looks at) and level 1
    // (slots past the end of the stretch become dead tokens, spread over the bins of 32 octaves: see slice_count_and_stash)
    const Frame fr = frame_of(M, eb);
    const uint32_t mine = uniform(g_end - min((uint32_t)wave * G, g_end));          // groups of the wave's stretch
    // (the mask is made opaque, so that the fractions are not kept, a register each, for the levels and the weights further down)
    uint32_t fmask0 = 0x7FFFFFu;
    asm volatile("" : "+s"(fmask0));
    const float dead = (__builtin_fabsf(M) <= 100.0f ? M : 0.0f) - 48.0f - (float)(lane & 31);
#pragma unroll
    for (int j = 0; j < kRowR; ++j) {
        if ((uint32_t)(j * kWave) >= mine) {             // nothing of the row (a scalar test)
            eb[j * 4] = 0; eb[j * 4 + 1] = 0; eb[j * 4 + 2] = 0; eb[j * 4 + 3] = 0;
            continue;
        }
        if ((uint32_t)(j + 1) * (uint32_t)kWave > mine) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if ((uint32_t)(j * kWave + lane) >= mine) eb[j * 4 + q] = __float_as_uint(dead);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t b = fr.raw(__uint_as_float(eb[j * 4 + q]));
            eb[j * 4 + q] = b;
            atomicAdd(reinterpret_cast<unsigned long long *>(&L.hr8[(b >> 21) * 8u + (uint32_t)(lane & 7)]),
                      (unsigned long long)(kPackOne | (b & fmask0)));
        }
    }
    if (p.e_bits) {
        // diagnostics: e of every token, dead tokens as 0
        uint4 *dst = reinterpret_cast<uint4 *>(p.e_bits + (int64_t)row * p.V);
        auto live = [](uint32_t b) { return b < kEMinBits ? 0u : b; };
#pragma unroll
        for (int j = 0; j < kRowR; ++j)
            if (g0 + (uint32_t)(j * kWave) < g_end)
                dst[g0 + (uint32_t)(j * kWave)] = make_uint4(live(eb[j * 4]), live(eb[j * 4 + 1]), live(eb[j * 4 + 2]), live(eb[j * 4 + 3]));
    }
    __syncthreads();
    if (tid < kNB) {
        uint64_t w = 0;
        if (tid >= (int)kBin0) {
#pragma unroll
            for (int c = 0; c < 8; ++c) w += L.hr8[tid * 8 + c];
        }
        s.g[tid] = w;
    }
    __syncthreads();
    const uint64_t top_k = (uint64_t)p.top_k;
    Found f = hist_find_level1<false, LdsRowS>(s, top_k, p.top_p, lane, wave);
    // (what is the same for all threads stays in scalar registers, or in LDS until it is used)
    f.bin = uniform(f.bin); f.cnt_above = uniform(f.cnt_above); f.cnt_bin = uniform(f.cnt_bin);
    auto target = [&](uint32_t thr, uint32_t n_gt, uint32_t n_eq, u128 above, uint32_t rounds) {
        return target_of_wave(p, row, p.inj_u ? 0ull : L.rand64, xmax, s.D, s.P, thr, n_gt, n_eq, above, rounds, lane == 0);
    };

    // one tie of all the row's tokens: as on the streaming path
    if (f.cnt_bin == (uint32_t)p.V && bin_is_one_tie(s.g[f.bin], f.bin, e_bits_of(xmax, M))) {
        if (wave == 0) {
            const uint32_t thr1 = e_bits_of(xmax, M);
            const Target tg = target(thr1, 0u, f.cnt_bin, (u128)0, 0u);
            uint32_t lo_i = 0, hi_i = (uint32_t)p.V - 1u;
            while (lo_i < hi_i) {
                const uint32_t mid = (lo_i + hi_i) >> 1;
                if ((u128)(mid + 1u) * tg.w_tie >= tg.r) hi_i = mid; else lo_i = mid + 1u;
            }
            p.out[row] = (int32_t)lo_i;
            if (p.diag) p.diag[row].index = (int32_t)lo_i;
        }
        return;
    }

    // ---- the threshold: radix selection on the registers, 7 bits a level ----
    const uint32_t exb = f.bin >> 2;
    uint32_t lo = f.bin << 21, span = (1u << 21) - 1u;
    bool one_tie = false;
    if (f.cnt_bin > 1u && f.cnt_above == 0u) {
        // a boundary bin that is one tie of the row's largest token: no further level needed, and counting
        // it would queue its tokens up at one address
        const uint32_t emax = e_bits_of(xmax, M);
        one_tie = bin_is_one_tie(s.g[f.bin], f.bin, emax);
        if (one_tie) { lo = emax; span = 0u; }
    }
    // A moderate number of tokens at or above the boundary bin: every wave lists its own, bits of e and place in its
    // stretch, and everything behind -- the levels, the sums of the pick -- reads a few list entries per thread instead
    // of the registers (the first pass of the pick alone takes 15 instructions per token, listing some 4).  Up to a sixth of
    // the row, that is: where more is kept the lists themselves cost as much as the registers (1024 rows of 8192, more
    // than half of each kept: 28 us from the registers, 38 from lists).  512 x 32768 float16, 4 % kept: 31.3 -> 26.8
    // us a call; 512 x 50304: 55.5 -> 46.3; 200 x 50304: 27.6 -> 22.9; flat rows with top_k 1000, 512 x 32768: 38.3 -> 30.4.
    // (The bits are copied out of the compiler's sight: it kept what it had worked out from them in 200 registers.)
    uint64_t *kept = L.hr8 + (uint32_t)wave * kRowKeptW;             // (in no order)
    uint32_t nkept = 0u;
    const uint32_t bin_lo = f.bin << 21;
    const uint32_t at_or_above = f.cnt_above + f.cnt_bin;
    bool have_kept = at_or_above <= kRowKept && at_or_above * 6u <= (uint32_t)p.V;
    if (have_kept) {
        // (The groups of four that hold such a token first, side by side, and of 64 of these at a time their tokens: with votes about every token
        // 512 x 32768 float16, 4 % kept, took 26.8 us, like this 25.9.)
        uint32_t staged = 0u, done = 0u;                             // groups of the wave
        uint4 *ring = stage.grp[wave];
        uint32_t *where = stage.at[wave];
        auto take = [&](const uint32_t n) __attribute__((always_inline)) {           // the tokens of the next n <= 64 groups
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            const uint32_t i = (done + (uint32_t)lane) & (kRowStage - 1u);
            const uint4 g = ring[i];
            const uint32_t at4 = where[i], b4[4] = {g.x, g.y, g.z, g.w};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const bool in = (uint32_t)lane < n && b4[q] >= bin_lo;
                const uint64_t cand = __builtin_amdgcn_ballot_w64(in);
                const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(cand >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)cand, nkept));
                if (in && at < kRowKeptW) kept[at] = ((uint64_t)b4[q] << 32) | (at4 + (uint32_t)q);
                nkept += (uint32_t)__builtin_popcountll(cand);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            done += n;
        };
        uint32_t lane4 = (uint32_t)lane * 4u;
#pragma unroll
        for (int j = 0; j < kRowR; ++j) {
            uint32_t b0 = eb[j * 4], b1 = eb[j * 4 + 1], b2 = eb[j * 4 + 2], b3 = eb[j * 4 + 3];
            asm volatile("" : "+s"(staged), "+v"(lane4), "+v"(b0), "+v"(b1), "+v"(b2), "+v"(b3));
            const bool in = max(max(b0, b1), max(b2, b3)) >= bin_lo;
            const uint64_t cand = __builtin_amdgcn_ballot_w64(in);
            const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(cand >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)cand, staged)) & (kRowStage - 1u);
            if (in) { ring[at] = make_uint4(b0, b1, b2, b3); where[at] = lane4 + (uint32_t)(j * 256); }
            staged += (uint32_t)__builtin_popcountll(cand);
            if (staged - done >= (uint32_t)kWave) take((uint32_t)kWave);
        }
        if (staged != done) take(staged - done);
        if (nkept > kRowKeptW && lane == 0) L.nokept = 1u;
        __syncthreads();
        have_kept = L.nokept == 0u;
    }
    if (have_kept) {
        // fn(bits of e, place in the wave's stretch) for the wave's listed tokens
        auto listed = [&](auto fn) {
            for (uint32_t i = (uint32_t)lane; i < nkept; i += (uint32_t)kWave) {
                const uint64_t e = kept[i];
                fn((uint32_t)(e >> 32), (uint32_t)e);
            }
        };
        // Levels while there are more than a few tokens in the boundary bin, each in words of its own (cleared at the start) and looked at where they were
        // counted; of the few the first wave ranks every one against every other.  (Down to a single token, a level taking four barriers instead of two
        // and its single token a fifth: 512 x 32768 float16 25.9 us, like this 24.3.)
        for (uint32_t lv = 2; lv <= (uint32_t)kLevels && !one_tie && f.cnt_bin > kRowFew; ++lv) {
            const uint32_t dsh = level_shift(lv);
            uint64_t *hist = L.lev + (lv - 2u) * 128u;
            listed([&](uint32_t b, uint32_t) {
                if (b - lo <= span) atomicAdd(reinterpret_cast<unsigned long long *>(&hist[(b >> dsh) & 127u]), (unsigned long long)(kPackOne | (b & 0x7FFFFFu)));
            });
            __syncthreads();
            f = hist_find128(s, hist, f.cnt_above, f.mass_above, top_k, exb, lane, wave);
            lo |= f.bin << dsh;
            span = (1u << dsh) - 1u;
        }
        if (span != 0u) {
            listed([&](uint32_t b, uint32_t) {
                if (b - lo <= span) L.small[atomicAdd(&L.nsmall, 1u) & (kRowFew - 1u)] = b;
            });
            __syncthreads();
        }
        if (wave == 0) {
            uint32_t t = lo, n_gt = f.cnt_above, n_eq = f.cnt_bin;
            M96 above = uniform(m96(f.mass_above));
            if (span != 0u) {
                // (the largest is always kept: what is above the bin is not enough)
                const uint32_t n = min(uniform(f.cnt_bin), kRowFew), b = (uint32_t)lane < n ? L.small[lane] : 0u;
                uint32_t larger = 0, sum = 0;
                for (uint32_t k = 0; k < n; ++k) {
                    const uint32_t o = lane_of(b, k);
                    larger += o > b ? 1u : 0u;
                    sum += o > b ? (o & 0x7FFFFFu) | 0x800000u : 0u;
                }
                const uint64_t need = need_of(uniform(m96(s.P)), above, exb);
                const bool in = (uint32_t)lane < n && n_gt + larger < (uint32_t)min(top_k, (uint64_t)0xFFFFFFFFull) && sum < need;
                t = ~wave_max_u32(in ? ~b : 0u);
                const uint64_t at = __builtin_amdgcn_ballot_w64(in && b == t);
                const uint32_t l = (uint32_t)__builtin_ctzll(at);
                n_eq = (uint32_t)__builtin_popcountll(at); n_gt += lane_of(larger, l);
                above = above + mass_of((uint64_t)lane_of(sum, l), exb);
            }
            const Target tg = target(t, n_gt, n_eq, wide(above), kRowRounds);
            s.bc64[1] = tg.w_tie; s.bc128[0] = tg.r; s.bc32[6] = t;
        }
        __syncthreads();
        const uint32_t thr = uniform(s.bc32[6]);
        const uint64_t w_tie = s.bc64[1];
        const u128 r = s.bc128[0];
        auto weight = [=](uint32_t b) -> uint64_t { return (b > thr) ? w_of_bits(b) : (b == thr ? w_tie : 0ull); };
        uint64_t a = 0, h = 0;                           // halves summed apart
        listed([&](uint32_t b, uint32_t) { const uint64_t w = weight(b); a += w & 0xFFFFFFFFull; h += w >> 32; });
        a = wave_sum(a); h = wave_sum(h);
        if (lane == 0) L.wq[wave] = (u128)a + ((u128)h << 32);
        __syncthreads();
        // every wave looks which stretch holds the target (1 <= r <= the sum of all kept weights); that wave goes on
        const u128 wt = lane < kRowW ? L.wq[lane] : (u128)0, winc = wave_inclusive_scan(wt);
        const uint32_t wstar = (uint32_t)__builtin_ctzll(__builtin_amdgcn_ballot_w64(winc >= r));
        if ((uint32_t)wave != wstar) return;
        u128 rl = r - wide(lane_of(m96(winc - wt), wstar));
        // the wave's stretch in 64 pieces of 64 tokens, one per lane, then the tokens of one piece  (16 groups of 256, four to a lane: 0.25 us more)
        auto in_order = []() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
        L.lev[lane] = 0ull; L.lev[kWave + lane] = 0ull;
        in_order();
        listed([&](uint32_t b, uint32_t place) {
            const uint64_t w = weight(b);
            atomicAdd(reinterpret_cast<unsigned long long *>(&L.lev[place >> 6]), (unsigned long long)(w & 0xFFFFFFFFull));
            atomicAdd(reinterpret_cast<unsigned long long *>(&L.lev[(uint32_t)kWave + (place >> 6)]), (unsigned long long)(w >> 32));
        });
        in_order();
        const u128 gm = (u128)L.lev[lane] + ((u128)L.lev[kWave + lane] << 32), ginc = wave_inclusive_scan(gm);
        const uint32_t piece = (uint32_t)__builtin_ctzll(__builtin_amdgcn_ballot_w64(ginc >= rl));       // there is one
        rl -= wide(lane_of(m96(ginc - gm), piece));
        in_order();
        L.lev[lane] = 0ull;
        in_order();
        listed([&](uint32_t b, uint32_t place) { if (place >> 6 == piece) L.lev[place & 63u] = weight(b); });
        in_order();
        const u128 own = (u128)L.lev[lane], inc = wave_inclusive_scan(own);
        if (inc - own < rl && rl <= inc) {               // exactly one lane
            const int32_t idx = (int32_t)((uint32_t)wave * G * 4u + piece * (uint32_t)kWave + (uint32_t)lane);
            p.out[row] = idx;
            if (p.diag) p.diag[row].index = idx;
        }
        return;
    }
    // The tokens of the boundary bin are listed while level 2 counts them (where the bin's copies were: they
    // are done with), every wave its own in a list of its own -- no counter to share, no wait: the place is
    // the wave's running count plus the lane's rank among the wave's candidates of that instruction -- if
    // the bin holds few enough for every wave's share to fit; levels 3 and 4 then read the lists, a few
    // entries per thread, and not the registers again.  A wave whose share does not fit after all (a sorted
    // row: the whole bin in one stretch) says so, and the levels go on from the registers.
    uint32_t *list = reinterpret_cast<uint32_t *>(L.hr8) + (uint32_t)wave * kRowListW;
    const bool use_list = f.cnt_bin <= kRowList;
    bool have_list = false;
    uint32_t nlist = 0u;                                 // wave-uniform
    for (uint32_t lv = 2; lv <= (uint32_t)kLevels && !one_tie && f.cnt_bin > 1u; ++lv) {
        const uint32_t dsh = level_shift(lv);
        if (tid < 128 * 4) L.lev[tid] = 0;
        __syncthreads();
        // the mask is made opaque so that the 64 words to add are built here, level by level, and not
        // kept in 128 registers across the levels
        uint32_t fmask = 0x7FFFFFu;
        asm volatile("" : "+v"(fmask));
        if (use_list && lv == 2u) {                      // count and list
#pragma unroll
            for (int j = 0; j < kRowR; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t b = eb[j * 4 + q];
                    const bool in = b - lo <= span;
                    const uint64_t cand = __builtin_amdgcn_ballot_w64(in);
                    if (in) {
                        atomicAdd(reinterpret_cast<unsigned long long *>(&L.lev[((b >> dsh) & 127u) * 4u + (uint32_t)(lane & 3)]),
                                  (unsigned long long)(kPackOne | (b & fmask)));
                        const uint32_t at = nlist + __builtin_amdgcn_mbcnt_hi((uint32_t)(cand >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)cand, 0u));
                        if (at < kRowListW) list[at] = b;
                    }
                    nlist += (uint32_t)__builtin_popcountll(cand);
                }
            if (nlist > kRowListW && lane == 0) L.nolist = 1u;
        } else if (!have_list) {                         // count, from the registers
#pragma unroll
            for (int j = 0; j < kRowR; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t b = eb[j * 4 + q];
                    if (b - lo <= span)
                        atomicAdd(reinterpret_cast<unsigned long long *>(&L.lev[((b >> dsh) & 127u) * 4u + (uint32_t)(lane & 3)]),
                                  (unsigned long long)(kPackOne | (b & fmask)));
                }
        } else {
            for (uint32_t i = (uint32_t)lane; i < nlist; i += (uint32_t)kWave) {
                const uint32_t b = list[i];
                if (b - lo <= span)
                    atomicAdd(reinterpret_cast<unsigned long long *>(&L.lev[((b >> dsh) & 127u) * 4u + (uint32_t)(lane & 3)]),
                              (unsigned long long)(kPackOne | (b & fmask)));
            }
        }
        __syncthreads();
        if (lv == 2u) have_list = use_list && L.nolist == 0u;
        if (tid < 128) s.hm[tid] = L.lev[tid * 4] + L.lev[tid * 4 + 1] + L.lev[tid * 4 + 2] + L.lev[tid * 4 + 3];
        __syncthreads();
        f = hist_find128(s, s.hm, f.cnt_above, f.mass_above, top_k, exb, lane, wave);
        lo |= f.bin << dsh;
        span = (1u << dsh) - 1u;
    }
    if (span != 0u) {                                    // a single token left in the range: the threshold itself
        if (have_list) {
            for (uint32_t i = (uint32_t)lane; i < nlist; i += (uint32_t)kWave)
                if (list[i] - lo <= span) s.bc32[6] = list[i];
        } else {
#pragma unroll
            for (int j = 0; j < kRowR; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (eb[j * 4 + q] - lo <= span) s.bc32[6] = eb[j * 4 + q];
        }
        __syncthreads();
        lo = s.bc32[6];
    }
    const uint32_t thr = lo;
    if (wave == 0) {
        const Target tg = target(thr, f.cnt_above, f.cnt_bin, f.mass_above, kRowRounds);
        s.bc64[1] = tg.w_tie; s.bc128[0] = tg.r;
    }
    __syncthreads();
    const uint64_t w_tie = s.bc64[1];
    const u128 r = s.bc128[0];

    // ---- the pick: kept weights in index order.  Every wave sums its stretch, a quarter of its groups at a
    // time; the wave whose stretch holds the target then finds it alone, in one quarter. ----
    constexpr int qb[5] = {0, (kRowR + 3) / 4, (2 * kRowR + 3) / 4, (3 * kRowR + 3) / 4, kRowR};
    // few kept tokens (f.cnt_above of them and f.cnt_bin ties): groups of four without one are skipped a wave at a time
    // (fewer than one kept token per wave and group on average: where most groups hold one the test only costs)
    const bool sparse = (uint64_t)(f.cnt_above + f.cnt_bin) * 256u < (uint64_t)(uint32_t)p.V;
    // (here a tie counts with the full weight of the threshold, and what the ties of the thread have too
    // much, tie_less each, is taken off the sum: a select less per token)
    auto weight = [=](uint32_t b) -> uint64_t {
        const uint32_t x = b >= thr ? ((b & 0x7FFFFFu) | 0x800000u) : 0u;
        return (uint64_t)x << (((b >> 23) - 87u) & 63u);
    };
    const uint64_t tie_less = w_of_bits(thr) - w_tie;    // w_tie <= the weight of the threshold
    u128 wtot = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        u128 mine = 0;
        uint32_t ties = 0u;
#pragma unroll
        for (int j = qb[q]; j < qb[q + 1]; ++j) {
            if (sparse) {
                const uint32_t m4 = max(max(eb[j * 4], eb[j * 4 + 1]), max(eb[j * 4 + 2], eb[j * 4 + 3]));
                if (__builtin_amdgcn_ballot_w64(m4 >= thr) == 0ull) continue;
            }
            mine += (u128)weight(eb[j * 4]) + weight(eb[j * 4 + 1]) + weight(eb[j * 4 + 2]) + weight(eb[j * 4 + 3]);
            ties += (uint32_t)(eb[j * 4] == thr) + (uint32_t)(eb[j * 4 + 1] == thr) + (uint32_t)(eb[j * 4 + 2] == thr) + (uint32_t)(eb[j * 4 + 3] == thr);
            // four weights at a time: the running sum is made opaque, or all the weights are worked out first
            // (two registers each) and summed as a tree
            uint64_t lo64 = (uint64_t)mine, hi64 = (uint64_t)(mine >> 64);
            asm volatile("" : "+v"(lo64), "+v"(hi64));
            mine = ((u128)hi64 << 64) | lo64;
        }
        mine -= (u128)ties * tie_less;
        const u128 t = wave_sum(mine);
        if (lane == 0) L.wq4[wave][q] = t;
        wtot += t;
    }
    if (lane == 0) L.wq[wave] = wtot;
    __syncthreads();
    if (wave == 0) {                                     // 1 <= r <= the sum of all kept weights: one stretch holds it
        const u128 t = lane < kRowW ? L.wq[lane] : (u128)0;
        const u128 inc = wave_inclusive_scan(t);
        const u128 exc = inc - t;
        if (lane < kRowW && exc < r && r <= inc) { s.bc32[7] = (uint32_t)lane; s.bc128[1] = r - exc; }
    }
    __syncthreads();
    if (wave != (int)s.bc32[7]) return;
    u128 rl = s.bc128[1];                                // 1 <= rl <= the kept weight of this wave's stretch
    int qstar = 0;
    for (int q = 0; q < 3; ++q) { const u128 t = L.wq4[wave][q]; if (rl > t) { rl -= t; qstar = q + 1; } else break; }
    const int jlo = qb[qstar], jhi = qb[qstar + 1];
    // (The weights are worked out again, from copies of the bits the compiler cannot see through: kept from
    // the first time they would fill 128 registers.)
    auto weight2 = [=](uint32_t b) -> uint64_t {
        asm volatile("" : "+v"(b));
        return (b > thr) ? w_of_bits(b) : (b == thr ? w_tie : 0ull);
    };
    bool found = false;
#pragma unroll
    for (int j = 0; j < kRowR; ++j) {
        if (found || j < jlo || j >= jhi) continue;
        const u128 w0 = weight2(eb[j * 4]), w1 = weight2(eb[j * 4 + 1]), w2 = weight2(eb[j * 4 + 2]), w3 = weight2(eb[j * 4 + 3]);
        const u128 m4 = w0 + w1 + w2 + w3;
        const u128 inc = wave_inclusive_scan(m4);
        const u128 t = lane63(inc);
        if (rl > t && j < jhi - 1) { rl -= t; continue; }
        found = true;
        const u128 exc = inc - m4;
        if (exc < rl && rl <= inc) {                     // exactly one lane
            const u128 rr = rl - exc;                    // 1 <= rr <= m4
            const int kk = (rr <= w0) ? 0 : (rr <= w0 + w1) ? 1 : (rr <= w0 + w1 + w2) ? 2 : 3;
            const int32_t idx = (int32_t)((g0 + (uint32_t)(j * kWave)) * 4u + (uint32_t)kk);
            p.out[row] = idx;
            if (p.diag) p.diag[row].index = idx;
        }
    }
}

}  // namespace rs
