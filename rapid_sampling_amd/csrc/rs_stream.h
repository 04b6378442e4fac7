// The streaming path: one wait-free pass over the logits, a finishing workgroup per row.
#pragma once

#include "rs_common.h"
#include "rs_cluster.h"
#include "rs_mass.h"

namespace rs {

// ---------------------------------------------------------- streaming path --
// When the kept set is small next to the row the cluster kernel's exchanges
// cost more than the data movement.  The streaming path has no waits at all:
//
//   stream_kernel   one workgroup per slice.  It reads the slice once, takes
//                   its OWN maximum as the frame (the significand of e does
//                   not depend on the frame, so a slice's histogram is the
//                   row's up to a shift of whole octaves), adds its level-1
//                   histogram to the row's and stashes its largest tokens --
//                   several times its share of the row's top_k -- ordered by
//                   bin, with the exact value down to which the stash is
//                   complete.
//   finish_kernel   one workgroup per row.  It brings the row's histogram into
//                   the row's frame, finds the boundary bin, pulls the stashed
//                   tokens at or above it (or, for flat rows, the stashes
//                   whole), resolves the threshold on them and picks.  A row
//                   that cannot be finished from the stashes (a huge tie, a
//                   nucleus of thousands of tokens) it does alone, from the
//                   logits (finish_row_slow).
// For a call that keeps every live token (top_k = V, top_p = 1) the pass (KEEP) stops behind the histogram
// and leaves each slice's mass, one sum for every distance its frame may lie below the row's, where the
// stash would begin; keep_finish_kernel picks the slice from those and reads that one slice again.
// Lanes of a wave that add to one LDS address are served one after the other, and rows often put
// most of their tokens into a few bins.  So each bin is kept in kRep copies (lane l adds to copy
// l % kRep), and e is not clamped before it is counted: the histogram spans all 512 values of
// bits >> 21, the dead tokens (below 2^-40, often most of a row) spread over the bins below
// kBin0 by their own exponents, where nobody looks at them again.  The histogram is done with
// before the candidates are staged, and shares their memory.
// Eight copies for long slices; four for the middle ones, which keeps their histogram smaller than
// the candidate staging it shares memory with (six workgroups per CU); two for the short slices of
// small calls, where clearing and folding the copies would cost more than the few tokens of a thread.
template <int R> constexpr int stream_copies() { return R > 8 ? 8 : R == 8 ? 4 : 2; }
template <int kRep>
struct LdsA {
    union {
        uint64_t hm[kNB * kRep];     // the slice's bins by bits >> 21
        struct {
            uint4    grp[kStashCap];     // float4 groups that hold a candidate: bits of their 4 tokens
            uint32_t gidx[kStashCap];    // and the index of their first token
        };
    };
    uint32_t off[kSB];
    uint32_t sub[128];           // level-2 counts inside a boundary bin too large for the stash
    uint32_t u32[16];
    uint32_t n, cut, over;
};

#ifndef RS_STREAM_WAVES
#define RS_STREAM_WAVES 3
#endif
// Stores of per-slice data: plain for the streaming path of separate launches (the kernel boundary makes
// them visible), device-scope atomic stores for the one-launch path, whose finishing workgroup
// reads them while the kernel is still running.
template <bool FUSED, typename T> __device__ __forceinline__ void put(T *p, T v)
{
    if (FUSED) a_store(p, v); else *p = v;
}
template <bool FUSED, typename T> __device__ __forceinline__ T get(const T *p)
{
    if (FUSED) return a_load(p); else return *p;
}

// One slice of the streaming pass, from the scaled logits in the registers (eb: x of this thread's
// 4R tokens, lmax their maximum) to its published record: the slice's frame, e in that frame (left
// in eb), the packed histogram added to the row's and kept under the slice's own name, cumulative
// counts, and the stash of its largest tokens with the value down to which it is complete.
// Returns the key of the slice's maximum.
// KEEP: a call that keeps every live token (top_k = V, top_p = 1); kCap: room of the stash; PAD: slots past the end of the row
// are looked for (the host's rule, rs_stream.hip).
template <int R, int NT, int kRep, bool FUSED, bool KEEP = false, int kCap = kStashCap, bool PAD = false>
__device__ __forceinline__ uint32_t slice_count_and_stash(const Params &p, const StreamView &v, LdsA<kRep> &s, uint32_t (&eb)[R * 4],
                                                          const float lmax, const uint32_t row, const uint32_t part,
                                                          const uint32_t base4, const int nv)
{
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    const uint32_t G = v.G;
    {
        uint4 *z = reinterpret_cast<uint4 *>(&s.hm[kBin0 * kRep]);               // two words per store; the bins of dead tokens are never read
        constexpr int kWords = (kNB - (int)kBin0) * kRep / 2;
#pragma unroll
        for (int i = 0; i < (kWords + NT - 1) / NT; ++i)
            if ((i + 1) * NT <= kWords || tid + i * NT < kWords) z[tid + i * NT] = make_uint4(0u, 0u, 0u, 0u);
    }
    uint32_t k = wave_max_u32(fkey(lmax));
    if (lane == 0) s.u32[wave] = k;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < (NT / kWave); ++w) k = max(k, s.u32[w]);
    const float M = __builtin_floorf(fkey_inv(k));

    // e in the slice's frame, not yet clamped at 2^-40, and its histogram.  Slots past the end of the row are in its last slice
    // only.  A wave is spared them kChunk groups at a time, by a scalar test, where there is nothing of the row in any; those beside
    // live tokens become dead ones, spread over the bins of 32 octaves.  (A test per group and lane, slots left out one by one,
    // keeps the groups' instructions apart: 256 x 151936 bfloat16 32.6 us a call against 31.2, 64 x 152064 bfloat16, in slices of 8192
    // tokens, 18.9 against 18.3.)  In slices of 8192 tokens four groups at a time: all eight at once take 82 registers instead of 74, with
    // which five workgroups share a compute unit and not six, and calls of 1281 to 1536 of them need another round (512 x 20480 with
    // top_k 1000 43.1 us a call against 39.9).  Slices of 4096 tokens are tested, two groups at a time, in calls of more workgroups than compute
    // units (PAD): 300 x 16388 15.1 us a call against 16.1, 100 x 50304 14.4 against 14.9; a call whose workgroups have a compute unit each waits for
    // one chain, which the tests make longer (1 x 262144 10.43 with none, 10.51).  Slices of 16384 tokens are not tested at all unless a
    // quarter of the call's slots lie past the end of their rows (PAD, too): the tests cost such a call 1 % (512 x 50304, 23 % of the slots, 34.9 us a call without,
    // 35.2 with), the slots 2 to 8 % (1024 x 8196 25.1 and 23.2, 512 x 32772 with top_k 1000 51.7 and 50.5).
    // Calls that keep every token, which have no stash to select, hide the test per lane behind their loads and lose more by the registers
    // of groups that are worked out together: 512 x 50304 bfloat16, in slices of 8192, 27.2 us a call against 28.6 with one test of all eight,
    // in shorter slices nothing tested 10.4 against 10.5 (32 x 65536 bfloat16).
    const Frame fr = frame_of(M, eb);
    constexpr bool kLane = KEEP && R == 8;
    constexpr int kChunk = kLane ? 1 : PAD ? 2 : R == 8 && !FUSED ? 4 : R;
    constexpr bool kSkip = PAD || (R == 8 && !FUSED && !KEEP);   // (the one-launch kernel: 0.6 % slower with them over 92 shapes)
    const uint32_t first = uniform(base4), left = ((uint32_t)p.V >> 2) - min(first, (uint32_t)p.V >> 2);      // groups of the row from the wave's first one on
    const float dead = (__builtin_fabsf(M) <= 100.0f ? M : 0.0f) - 48.0f - (float)(lane & 31);
#pragma unroll
    for (int jc = 0; jc < R; jc += kChunk) {
        if (kLane ? jc >= nv : kSkip && (uint32_t)(jc * NT) >= left) {
#pragma unroll
            for (int i = jc * 4; i < (jc + kChunk) * 4; ++i) eb[i] = 0;
            continue;
        }
        if (!kLane && (uint32_t)((jc + kChunk - 1) * NT + kWave) > left) {
#pragma unroll
            for (int j = jc; j < jc + kChunk; ++j)
                if (j >= nv) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) eb[j * 4 + q] = __float_as_uint(dead);
                }
        }
#pragma unroll
        for (int i = jc * 4; i < (jc + kChunk) * 4; ++i) {
            const uint32_t b = fr.raw(__uint_as_float(eb[i]));
            eb[i] = b;
            atomicAdd(reinterpret_cast<unsigned long long *>(&s.hm[(b >> 21) * kRep + (lane & (kRep - 1))]),
                      (unsigned long long)(kPackOne | (b & 0x7FFFFFu)));
        }
    }
    if (p.e_bits) {
        // diagnostics: e of every token, still in the slice's frame; the finishing workgroup re-bases it
        uint4 *dst = reinterpret_cast<uint4 *>(p.e_bits + (int64_t)row * p.V);
#pragma unroll
        for (int j = 0; j < R; ++j)
            if (j < nv) {
                if (FUSED) {
                    uint32_t *w = reinterpret_cast<uint32_t *>(&dst[base4 + j * NT]);
                    a_store(&w[0], eb[j * 4]); a_store(&w[1], eb[j * 4 + 1]); a_store(&w[2], eb[j * 4 + 2]); a_store(&w[3], eb[j * 4 + 3]);
                } else dst[base4 + j * NT] = make_uint4(eb[j * 4], eb[j * 4 + 1], eb[j * 4 + 2], eb[j * 4 + 3]);
            }
    }
    __syncthreads();
    // Add the slice's live bins to the row's, which are kept by absolute octave (mod 128, 4 bins each):
    // bin t of this frame is octave M - 40 + t/4.  Slices of one row may use different frames; as
    // long as their maxima lie within 87 octaves of each other no two octaves in use coincide.
    auto bin_total = [&](int b) {
        const uint4 *two = reinterpret_cast<const uint4 *>(&s.hm[((int)kBin0 + b) * kRep]);     // two copies per load
        uint64_t w = 0;
#pragma unroll
        for (int c = 0; c < kRep / 2; ++c) {
            const uint4 q = two[c];
            w += (((uint64_t)q.y << 32) | q.x) + (((uint64_t)q.w << 32) | q.z);
        }
        return w;
    };
    const bool plain = KEEP && p.report == 0u;           // (not the first pass of the two-pass wide path)
    if (!plain && tid < kSB) {
        const uint64_t w = bin_total(tid);
        const float mm = M - 128.0f * __builtin_floorf(M * 0.0078125f);          // M mod 128, exact
        put<FUSED>(&v.shist[((size_t)row * G + part) * kSB + tid], w);          // kept for rows whose slices lie far apart
        uint64_t *rowbins = FUSED ? (p.ctl_end - 1 - row)->h[0] : (p.ctl_end - 1 - row)->rowhist;
        if (w) a_add(&rowbins[((uint32_t)(int)mm * 4u + (uint32_t)tid - 160u) & 511u], w);
    }
    if constexpr (KEEP) {
        // every live token is kept: what the finishing workgroup needs of this slice is its mass in the row's frame, which
        // may lie d octaves above this one's and leaves the lowest 4 d bins dead: the mass of the bins from 4 d on, for
        // every d, left where the stash would begin
        if (plain && wave == 0) {
            BinScan<3> sc;
            auto at = [&](int i) { return kSB - 1 - 3 * lane - i; };
            sc.load([&](int i) { return at(i) >= 0 ? bin_total(max(at(i), 0)) : 0ull; }, [&](int i) { return (kBin0 + (uint32_t)max(at(i), 0)) >> 2; });
            uint64_t *st = v.stash + ((size_t)row * G + part) * kStashCap;
            Limbs from = sc.mb;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                from = from + sc.m[i];
                if (at(i) >= 0 && (at(i) & 3) == 0) {
                    const M96 q = m96(from);
                    reinterpret_cast<uint4 *>(st)[at(i) >> 2] = make_uint4((uint32_t)q.lo, (uint32_t)(q.lo >> 32), q.hi, 0u);
                }
            }
        }
        if (tid == 0) {
            PartHdr ph;
            ph.mkey = k; ph.window = 0u; ph.n = 0u; ph.cut = 0u;
            v.hdr[(size_t)row * G + part] = ph;
        }
        return k;
    }

    // What to stash: the bins from the top down to the first one at which the count reaches
    // stash_k (that bin too if it fits).  With stash_k = top_k the row's top_k tokens are certainly
    // in the stashes; the host aims lower when a row has many slices, since a slice then holds
    // about top_k / slices of them, and the finishing workgroup checks that each stash reaches
    // down to the row's boundary bin before it relies on it.
    if (wave == 0) {
        const uint32_t Ks = p.stash_k;
        uint32_t c3[3];
        uint32_t cs = 0;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int b = kSB - 1 - 3 * lane - i;
            c3[i] = b >= 0 ? pack_count(bin_total(b)) : 0u;
            cs += c3[i];
        }
        const uint32_t ci = wave_inclusive_scan(cs);
        uint32_t run = ci - cs;
        const uint32_t total = lane63(ci);
        if (lane == 0) s.over = 0xFFFFFFFFu;
        if (lane == 0 && total < Ks) { s.n = total; s.cut = kBin0 << 21; }   // a short slice: all its live tokens
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int b = kSB - 1 - 3 * lane - i;
            const uint32_t nx = run + c3[i];
            if (b >= 0) {
                s.off[b] = run;                                           // tokens in the bins above b
                put<FUSED>(&v.cum[((size_t)row * G + part) * kSB + b], nx);
            }
            if (run < Ks && nx >= Ks) {
                // the whole bin if that stays close to stash_k, else only part of it (found below)
                if (nx <= min((uint32_t)kCap, Ks + max(64u, Ks >> 2))) { s.n = nx; s.cut = ((uint32_t)b + kBin0) << 21; }
                else { s.n = run; s.cut = ((uint32_t)b + 1u + kBin0) << 21; s.over = (uint32_t)b; }
            }
            run = nx;
        }
    }
    if (tid < 128) s.sub[tid] = 0;
    __syncthreads();
    if (s.over != 0xFFFFFFFFu) {
        // The bin in which the count reaches stash_k holds far more tokens than asked for (a flat
        // distribution: hundreds or thousands of tokens within a quarter octave).  Look at its next
        // 7 bits and take the sub-bins from the top down to the one at which the count reaches
        // stash_k, as far as they fit.
        const uint32_t ob = s.over + kBin0, above = s.n;
        // a bin that is one tie of the slice's largest token (rows of equal logits) has all its
        // tokens in one sub-bin: known without counting, which would queue them up at one address
        const uint32_t emax = e_bits_raw(fkey_inv(k), M);
        const uint64_t wbin = bin_total((int)s.over);
        if (above == 0u && bin_is_one_tie(wbin, ob, emax)) {
            if (tid == 0) s.sub[(emax >> 14) & 127u] = pack_count(wbin);
        } else {
#pragma unroll
            for (int j = 0; j < R; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t b = eb[j * 4 + q];
                    if ((b >> 21) == ob) atomicAdd(&s.sub[(b >> 14) & 127u], 1u);
                }
        }
        __syncthreads();
        if (wave == 0) {
            const uint32_t Ks = p.stash_k;
            const uint32_t c0 = s.sub[127 - 2 * lane], c1 = s.sub[126 - 2 * lane];
            const uint32_t ci = wave_inclusive_scan(c0 + c1);
            const uint32_t r0 = above + ci - c0 - c1, r1 = r0 + c0, r2 = r1 + c1;
            // first sub-bin at which the count reaches stash_k (there is one: the whole bin reaches it)
            if (r0 < Ks && r1 >= Ks) {
                const bool fits = r1 <= (uint32_t)kCap;
                s.n = fits ? r1 : r0;
                s.cut = (ob << 21) + ((127u - 2u * (uint32_t)lane + (fits ? 0u : 1u)) << 14);
            } else if (r1 < Ks && r2 >= Ks) {
                const bool fits = r2 <= (uint32_t)kCap;
                s.n = fits ? r2 : r1;
                s.cut = (ob << 21) + ((126u - 2u * (uint32_t)lane + (fits ? 0u : 1u)) << 14);
            }
        }
        __syncthreads();
    }
    const uint32_t n = s.n, cut = s.cut;
    // From here on the bits in the registers are compared with the cut, which is never below
    // 2^-40: dead tokens are no candidates.

    // Candidates (bits >= cut) are at most n <= kCap, so at most that many float4 groups
    // hold one.  Each thread copies its groups with a candidate into LDS at an offset from a scan
    // of the per-thread counts; the tokens of those groups are then gone through densely.
    uint32_t mine = 0;
#pragma unroll
    for (int j = 0; j < R; ++j)
        mine += max(max(eb[j * 4], eb[j * 4 + 1]), max(eb[j * 4 + 2], eb[j * 4 + 3])) >= cut ? 1u : 0u;
    uint32_t o = wave_inclusive_scan(mine);
    if (lane == kWave - 1) s.u32[wave] = o;
    __syncthreads();
    uint32_t ngroups = 0;
#pragma unroll
    for (int w = 0; w < (NT / kWave); ++w) {
        if (w < wave) o += s.u32[w];
        ngroups += s.u32[w];
    }
    o -= mine;
#pragma unroll
    for (int j = 0; j < R; ++j) {
        if (max(max(eb[j * 4], eb[j * 4 + 1]), max(eb[j * 4 + 2], eb[j * 4 + 3])) >= cut) {
            if (o < (uint32_t)kCap) {
                s.grp[o] = make_uint4(eb[j * 4], eb[j * 4 + 1], eb[j * 4 + 2], eb[j * 4 + 3]);
                s.gidx[o] = (base4 + (uint32_t)j * NT) * 4;
            }
            ++o;
        }
    }
    __syncthreads();
    // Write the candidates out grouped by bin, largest e first, so that the finishing
    // workgroup can take a prefix.
    uint64_t *st = v.stash + ((size_t)row * G + part) * kStashCap;
    const uint32_t *gb = reinterpret_cast<const uint32_t *>(s.grp);
#pragma unroll 4
    for (uint32_t i = tid; i < min(ngroups, (uint32_t)kCap) * 4u; i += NT) {
        const uint32_t b = gb[i];
        if (b >= cut) {
            const uint32_t slot = atomicAdd(&s.off[(b >> 21) - kBin0], 1u);
            if (slot < (uint32_t)kCap) put<FUSED>(&st[slot], ((uint64_t)b << 32) | (s.gidx[i >> 2] + (i & 3u)));
        }
    }
    if (tid == 0) {
        if (FUSED) {
            uint64_t *h2 = reinterpret_cast<uint64_t *>(&v.hdr[(size_t)row * G + part]);
            a_store(&h2[0], (uint64_t)k);
            a_store(&h2[1], ((uint64_t)cut << 32) | n);
        } else {
            PartHdr ph;
            ph.mkey = k; ph.window = 0u; ph.n = n; ph.cut = cut;
            v.hdr[(size_t)row * G + part] = ph;
        }
    }
    return k;
}

template <int R, int NT, int DT, bool KEEP = false, bool PAD = false>     // NT threads, each with R groups of four tokens of the slice; DT the logits' type
__global__ void __launch_bounds__(NT, (R <= 8 ? 5 : RS_STREAM_WAVES)) stream_kernel(const Params p, const StreamView v)
{
    constexpr int kRep = stream_copies<R>();
    __shared__ LdsA<kRep> s;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    const uint32_t G = v.G;
    const uint32_t row = blockIdx.x / G, part = blockIdx.x - row * G;
    const uint32_t V4 = (uint32_t)p.V >> 2;
    const uint32_t base4 = part * (uint32_t)(NT * R) + (uint32_t)tid;
    const int nv = base4 >= V4 ? 0 : (int)min((uint32_t)R, (V4 - base4 + NT - 1) / NT);
    const char *lrow = logits_row(p, row);

    const bool reporter = blockIdx.x == 0 && tid == 0;
    PrevCall prev;
    prev.slow_rows = 0; prev.meta = 0;
    if (reporter) prev = report_begin(p);
    uint32_t eb[R * 4];                                 // l, then x, then bits(e)
    // x = l * c is the definition unless a NaN or Inf shows up (see sample_kernel).  Slots past the
    // end of the row read its last group again: harmless for the maximum and the probe, and they
    // are set aside before the histogram.
    constexpr int kSpecial = 0x207;
    float probe = 0.0f;
    float lmax = -3.402823466e+38f;
    if constexpr (DT == RS_DTYPE_F32) {
        const float4 *lg = reinterpret_cast<const float4 *>(lrow);
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const uint4 l = load_once(reinterpret_cast<const uint4 *>(lg) + min(base4 + (uint32_t)(j * NT), V4 - 1));
            eb[j * 4 + 0] = l.x; eb[j * 4 + 1] = l.y; eb[j * 4 + 2] = l.z; eb[j * 4 + 3] = l.w;
        }
    } else {
        const uint2 *lh = reinterpret_cast<const uint2 *>(lrow);
        uint2 h[R];
#pragma unroll
        for (int j = 0; j < R; ++j) h[j] = load_once(lh + min(base4 + (uint32_t)(j * NT), V4 - 1));
#pragma unroll
        for (int j = 0; j < R; ++j) widen4(h[j], DT, &eb[j * 4]);
    }
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const float x0 = __uint_as_float(eb[j * 4]) * p.c, x1 = __uint_as_float(eb[j * 4 + 1]) * p.c;
        const float x2 = __uint_as_float(eb[j * 4 + 2]) * p.c, x3 = __uint_as_float(eb[j * 4 + 3]) * p.c;
        probe = __builtin_fmaf(x0, x1, probe);
        probe = __builtin_fmaf(x2, x3, probe);
        lmax = fmaxf(fmaxf(lmax, x0), fmaxf(x1, fmaxf(x2, x3)));
        eb[j * 4 + 0] = __float_as_uint(x0); eb[j * 4 + 1] = __float_as_uint(x1);
        eb[j * 4 + 2] = __float_as_uint(x2); eb[j * 4 + 3] = __float_as_uint(x3);
    }
    if (__builtin_amdgcn_classf(probe, kSpecial)) {
        // the clean-up of sampling.cu:553 on the products already in the registers (masked
        // vocabularies, logits at -inf, come through here on every call)
        lmax = -3.402823466e+38f;
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const float x0 = sf(__uint_as_float(eb[j * 4])), x1 = sf(__uint_as_float(eb[j * 4 + 1]));
            const float x2 = sf(__uint_as_float(eb[j * 4 + 2])), x3 = sf(__uint_as_float(eb[j * 4 + 3]));
            if (j < nv) lmax = fmaxf(lmax, fmaxf(fmaxf(x0, x1), fmaxf(x2, x3)));
            eb[j * 4 + 0] = __float_as_uint(x0); eb[j * 4 + 1] = __float_as_uint(x1);
            eb[j * 4 + 2] = __float_as_uint(x2); eb[j * 4 + 3] = __float_as_uint(x3);
        }
    }
    // a call that keeps everything has no rows to report on; the counting-only pass of the wide path does
    if (reporter) report_end(p, prev, !KEEP || p.report != 0u);
    slice_count_and_stash<R, NT, kRep, false, KEEP, kStashCap, PAD>(p, v, s, eb, lmax, row, part, base4, nv);
}

struct LdsB {
    uint64_t *list;              // gathered tokens, row frame: bits << 32 | index (dynamic LDS, v.list_cap entries)
    uint64_t blo[kMaxParts], bhi[kMaxParts];
    uint64_t small[64];
    uint32_t delta[kMaxParts];   // octaves between the row's frame and slice g's
    uint32_t m4[kMaxParts];      // 4 (M mod 128) of slice g's frame: where its bins sit among the row's positions
    uint32_t take[kMaxParts];    // inclusive prefix of the entries taken from each stash
    uint64_t rand64;
    struct { M96 D, P, above; uint32_t place, cnt_above, cnt_bin, found; } one;   // what one wave worked out for all (finish_row)
    uint32_t nsmall, bucket, fail;
    uint32_t result;             // sampled token + 1 once the row is finished
};

// The call's parameters, read from the kernel's arguments once more (they are the first of them in every kernel): for the
// ways that almost no row takes.  Otherwise what only those need is loaded at the kernel's start and kept, in scalar
// registers that the usual chain is short of: the finishing kernel of eight slices a wave spilled 36 of them, 7 this way, and
// over 192 shapes of 1 to 256 rows its calls take 0.991 of their time (64 rows of 152064 19.66 -> 19.26 us a call, of 65540 15.65 -> 15.31).
__device__ __forceinline__ Params params_again()
{
    auto *args = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    Params p;
    __builtin_memcpy(&p, (const void *)args, sizeof(Params));
    return p;
}

// A row the stashes cannot finish (a nucleus or a tie of thousands of tokens, more kept tokens than
// the list holds): the finishing workgroup does it alone, from the logits, in a few passes over the
// row -- the level-1 histogram in the row's frame (M = floor of the row's maximum is known), the
// next digits of the threshold inside the boundary bin until the bin's tokens fit a gathered list,
// the rest in LDS, then the inverse CDF by buckets of the token index, by sub-buckets, and token
// by token.  A few passes of one workgroup over one row take tens of microseconds (a row of a
// million tokens: more than a hundred): fine for the odd row, and calls whose rows mostly end here
// are routed to the cluster kernel by the caller's policy.  Same integers as every other path.
__device__ __forceinline__ void finish_row_slow(const Params &p, Lds &s, LdsB &t, const uint32_t row, const float xmax, const uint64_t rand64)
{
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    const uint32_t V4 = (uint32_t)p.V >> 2;
    const float M = __builtin_floorf(xmax);
    const char *lrow = logits_row(p, row);
    const float4 *pn4 = p.penalties ? reinterpret_cast<const float4 *>(p.penalties + (int64_t)row * p.V) : nullptr;
    // bits of e of four tokens, by the definition (reference: sampling.cu:220, :553)
    auto bits_of4 = [&](const float4 l, const float4 q) -> uint4 {
        float x0, x1, x2, x3;
        if (pn4) {
            x0 = sf((sf(l.x) - q.x) * p.c); x1 = sf((sf(l.y) - q.y) * p.c); x2 = sf((sf(l.z) - q.z) * p.c); x3 = sf((sf(l.w) - q.w) * p.c);
        } else {
            x0 = sf(l.x * p.c); x1 = sf(l.y * p.c); x2 = sf(l.z * p.c); x3 = sf(l.w * p.c);
        }
        return make_uint4(e_bits_of(x0, M), e_bits_of(x1, M), e_bits_of(x2, M), e_bits_of(x3, M));
    };
    // fn(token index, bits of its e) for the tokens of groups [lo4, hi4) of the row, four loads in flight per thread
    auto row_pass = [&](uint32_t lo4, uint32_t hi4, auto fn) {
        constexpr int kAhead = 4;
        for (uint32_t base = lo4 + (uint32_t)tid; base < hi4; base += kAhead * kThreads) {
            float4 l[kAhead], q[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const uint32_t i4 = min(base + (uint32_t)u * kThreads, hi4 - 1u);
                l[u] = load_logits4(lrow, i4, p.dtype);
                q[u] = pn4 ? pn4[i4] : make_float4(0.f, 0.f, 0.f, 0.f);
            }
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const uint32_t i4 = base + (uint32_t)u * kThreads;
                if (i4 < hi4) {
                    const uint4 b = bits_of4(l[u], q[u]);
                    fn(i4 * 4u, b.x); fn(i4 * 4u + 1u, b.y); fn(i4 * 4u + 2u, b.z); fn(i4 * 4u + 3u, b.w);
                }
            }
        }
    };
    const uint64_t top_k = (uint64_t)p.top_k;
    // level 1 (dead tokens, below 2^-40, are left out)
    __syncthreads();
    for (int b = tid; b < kNB * kRepC; b += kThreads) s.hr[b] = 0;
    __syncthreads();
    row_pass(0u, V4, [&](uint32_t, uint32_t b) {
        if (b >= kEMinBits)
            atomicAdd(reinterpret_cast<unsigned long long *>(&s.hr[(b >> 21) * kRepC + (lane & (kRepC - 1))]),
                      (unsigned long long)(kPackOne | (b & 0x7FFFFFu)));
    });
    __syncthreads();
    for (int b = tid; b < kNB; b += kThreads) {
        uint64_t w = 0;
#pragma unroll
        for (int c = 0; c < kRepC; ++c) w += s.hr[b * kRepC + c];
        s.g[b] = w;
    }
    __syncthreads();
    Found f = hist_find_level1<false>(s, top_k, p.top_p, lane, wave);
    const u128 D = s.D, P = s.P;
    const uint32_t exb = f.bin >> 2;
    uint32_t lo = f.bin << 21, span = (1u << 21) - 1u, levels = 1;
    bool one_tie = false;
    if (f.cnt_bin > (uint32_t)kCap && f.cnt_above == 0u) {
        const uint32_t emax = e_bits_of(xmax, M);
        one_tie = bin_is_one_tie(s.g[f.bin], f.bin, emax);
        if (one_tie) { lo = emax; span = 0u; }
    }
    // further digits over the whole row while the boundary bin holds more tokens than can be gathered
    while (!one_tie && f.cnt_bin > (uint32_t)kCap && levels < (uint32_t)kLevels) {
        ++levels;
        const uint32_t dsh = level_shift(levels);
        __syncthreads();
        lds_hist_zero(s, 128);
        __syncthreads();
        row_pass(0u, V4, [&](uint32_t, uint32_t b) {
            if (b - lo <= span) lds_hist_add(s, (b >> dsh) & 127u, b);
        });
        __syncthreads();
        f = hist_find128(s, s.hm, f.cnt_above, f.mass_above, top_k, exb, lane, wave);
        lo |= f.bin << dsh;
        span = (1u << dsh) - 1u;
    }
    if (f.cnt_bin <= (uint32_t)kCap) {
        // gather the bin's tokens and resolve the remaining digits on them
        __syncthreads();
        if (tid == 0) s.ctr = 0;
        __syncthreads();
        row_pass(0u, V4, [&](uint32_t idx, uint32_t b) {
            if (b - lo <= span) {
                const uint32_t o = atomicAdd(&s.ctr, 1u);
                if (o < (uint32_t)kCap) s.cand[o] = ((uint64_t)b << 32) | idx;
            }
        });
        __syncthreads();
        const uint32_t ncand = min(s.ctr, (uint32_t)kCap);
        for (uint32_t lv = levels + 1; lv <= (uint32_t)kLevels && f.cnt_bin > 1u && span != 0u; ++lv) {
            const uint32_t dsh = level_shift(lv);
            lds_hist_zero(s, 128);
            __syncthreads();
            for (uint32_t i = tid; i < ncand; i += kThreads) {
                const uint32_t b = (uint32_t)(s.cand[i] >> 32);
                if (b - lo <= span) lds_hist_add(s, (b >> dsh) & 127u, b);
            }
            __syncthreads();
            f = hist_find128(s, s.hm, f.cnt_above, f.mass_above, top_k, exb, lane, wave);
            lo |= f.bin << dsh;
            span = (1u << dsh) - 1u;
        }
        if (span != 0u) {
            for (uint32_t i = tid; i < ncand; i += kThreads) {
                const uint32_t b = (uint32_t)(s.cand[i] >> 32);
                if (b - lo <= span) s.bc32[6] = b;
            }
            __syncthreads();
            lo = s.bc32[6];
        }
    }
    const uint32_t thr = lo;
    if (tid == 0) {
        const Target tg = tie_and_target(p, row, rand64, xmax, D, P, thr, f.cnt_above, f.cnt_bin, f.mass_above, 8u, true);
        s.bc64[1] = tg.w_tie; s.bc128[0] = tg.r;
    }
    __syncthreads();
    const uint64_t w_tie = s.bc64[1];
    u128 r = s.bc128[0];
    auto weight = [&](uint32_t b) -> uint64_t { return (b > thr) ? w_of_bits(b) : (b == thr ? w_tie : 0); };

    // inverse CDF in index order: 256 buckets of 2^sh1 tokens, 256 sub-buckets of 2^sh2, then one by one
    uint32_t sh1 = 0;
    while (((uint32_t)p.V - 1u) >> sh1 >= 256u) ++sh1;
    const uint32_t sh2 = sh1 > 8u ? sh1 - 8u : 0u;
    auto bucket_pass = [&](uint32_t lo_idx, uint32_t hi_idx, uint32_t shift) -> uint32_t {
        t.blo[tid] = 0; t.bhi[tid] = 0;
        __syncthreads();
        const uint32_t a4 = lo_idx >> 2, e4 = min(V4, (hi_idx + 3u) >> 2);
        row_pass(a4, e4, [&](uint32_t idx, uint32_t b) {
            const uint64_t w = weight(b);
            if (w && idx >= lo_idx && idx < hi_idx) {
                const uint32_t bk = (idx - lo_idx) >> shift;               // < 256: the range spans at most 256 buckets
                atomicAdd(reinterpret_cast<unsigned long long *>(&t.blo[bk]), (unsigned long long)(w & 0xFFFFFFFFull));
                atomicAdd(reinterpret_cast<unsigned long long *>(&t.bhi[bk]), (unsigned long long)(w >> 32));
            }
        });
        __syncthreads();
        const u128 mine = (u128)t.blo[tid] + ((u128)t.bhi[tid] << 32);
        u128 inc = wave_inclusive_scan(mine);
        if (lane == kWave - 1) s.q128[wave] = inc;
        __syncthreads();
        for (int w = 0; w < wave; ++w) inc += s.q128[w];
        const u128 exc = inc - mine;
        if (exc < r && r <= inc) { t.bucket = (uint32_t)tid; s.bc128[1] = r - exc; }
        __syncthreads();
        r = s.bc128[1];
        const uint32_t bk = t.bucket;
        __syncthreads();
        return bk;
    };
    const uint32_t b1 = bucket_pass(0u, (uint32_t)p.V, sh1);
    uint32_t lo_idx = b1 << sh1;
    if (sh1 > sh2) {
        const uint32_t b2 = bucket_pass(lo_idx, min((uint32_t)p.V, lo_idx + (1u << sh1)), sh2);
        lo_idx += b2 << sh2;
    }
    if (tid == 0) {
        // the last few tokens one after the other
        const uint32_t hi_idx = min((uint32_t)p.V, lo_idx + (1u << sh2));
        uint32_t pick = lo_idx;
        u128 acc = 0;
        bool found = false;
        for (uint32_t i4 = lo_idx >> 2; i4 * 4u < hi_idx && !found; ++i4) {
            const uint4 b = bits_of4(load_logits4(lrow, i4, p.dtype), pn4 ? pn4[i4] : make_float4(0.f, 0.f, 0.f, 0.f));
            auto step = [&](uint32_t idx, uint32_t bits) {
                if (found || idx < lo_idx || idx >= hi_idx) return;
                acc += weight(bits);
                if (acc >= r) { pick = idx; found = true; }
            };
            step(i4 * 4u, b.x); step(i4 * 4u + 1u, b.y); step(i4 * 4u + 2u, b.z); step(i4 * 4u + 3u, b.w);
        }
        p.out[row] = (int32_t)pick;
        if (p.diag) p.diag[row].index = (int32_t)pick;
        t.result = pick + 1u;
    }
}

// The last step of the wide paths' finishes: the slice that begins at token lo_idx holds
// the target, r is the target's offset inside the slice.  The slice is gone through in chunks of
// 64 float4 groups (256 consecutive tokens, one KB that a wave loads in one go): chunk c belongs
// to wave c mod 4, which sums its tokens' weights (two 64-bit wave sums of the weights' halves);
// one wave scans the chunk totals for the chunk that holds the target, loads that chunk again,
// scans its 64 groups, and the lane whose group holds the target walks its four tokens.  No
// atomics, no list.  (An earlier version gave every thread 16 consecutive groups: its loads, 64
// cache lines per instruction and every line touched by 8 instructions, cost a microsecond per
// group.)  No penalties on this path.
// `kept`: what the threshold and the tie weight leave of a token's weight, from the bit pattern of its e in the
// row's frame.
template <int SLICE_LOG2, typename WF>
__device__ __forceinline__ void keep_pick(const Params &p, Lds &s, LdsB &t, const uint32_t row, const float M, const uint32_t lo_idx, const u128 r,
                                          WF kept)
{
    constexpr int N = 1 << (SLICE_LOG2 - 10);                      // chunks per wave
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    const uint32_t V4 = (uint32_t)p.V >> 2;
    const char *lrow = logits_row(p, row);
    const uint32_t g0 = lo_idx >> 2;
    auto weight = [&](float l) -> uint64_t { return kept(e_bits_of(sf(l * p.c), M)); };
    float4 l[N];
#pragma unroll
    for (int j = 0; j < N; ++j) l[j] = load_logits4(lrow, min(g0 + (uint32_t)((j * kWaves + wave) * kWave + lane), V4 - 1u), p.dtype);
#pragma unroll
    for (int j = 0; j < N; ++j) {
        uint64_t a = 0, b = 0;
        if (g0 + (uint32_t)((j * kWaves + wave) * kWave + lane) < V4) {            // past the end of the row: no weight
            const uint64_t w0 = weight(l[j].x), w1 = weight(l[j].y), w2 = weight(l[j].z), w3 = weight(l[j].w);
            a = (w0 & 0xFFFFFFFFull) + (w1 & 0xFFFFFFFFull) + (w2 & 0xFFFFFFFFull) + (w3 & 0xFFFFFFFFull);
            b = (w0 >> 32) + (w1 >> 32) + (w2 >> 32) + (w3 >> 32);
        }
        a = wave_sum(a); b = wave_sum(b);
        if (lane == 0) { t.blo[j * kWaves + wave] = a; t.bhi[j * kWaves + wave] = b; }
    }
    __syncthreads();
    if (wave == 0) {
        const u128 mine = lane < N * kWaves ? (u128)t.blo[lane] + ((u128)t.bhi[lane] << 32) : (u128)0;
        const u128 inc = wave_inclusive_scan(mine);
        const u128 exc = inc - mine;
        if (exc < r && r <= inc) { t.bucket = (uint32_t)lane; s.bc128[1] = r - exc; }
    }
    __syncthreads();
    if (wave == 0) {
        const uint32_t g = g0 + t.bucket * (uint32_t)kWave + (uint32_t)lane;
        const u128 r2 = s.bc128[1];
        uint64_t w[4] = {0ull, 0ull, 0ull, 0ull};
        if (g < V4) {
            const float4 q = load_logits4(lrow, g, p.dtype);
            w[0] = weight(q.x); w[1] = weight(q.y); w[2] = weight(q.z); w[3] = weight(q.w);
        }
        const u128 mine = (u128)w[0] + w[1] + w[2] + w[3];
        const u128 inc = wave_inclusive_scan(mine);
        u128 acc = inc - mine;
        if (acc < r2 && r2 <= inc) {
            uint32_t pick = g * 4u + 3u;
            bool found = false;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                acc += w[q];
                if (!found && acc >= r2) { pick = g * 4u + (uint32_t)q; found = true; }
            }
            p.out[row] = (int32_t)pick;
            if (p.diag) p.diag[row].index = (int32_t)pick;
            t.result = pick + 1u;
        }
    }
}

// Penalties at scale (stream_pen_kernel): the pass has already written every slice's decayed penalties and
// noted the old values that were not +0.0.  A row that has to be done the slow way needs the old values
// of all its tokens: the notes are played back, and every slice of the row is marked deferred, so that
// the fix-up kernel rewrites the whole row once its token is known.
__device__ __forceinline__ void pen_restore(const Params &p, const StreamView &v, const uint32_t row)
{
    const int tid = threadIdx.x;
    float *pen = p.penalties + (int64_t)row * p.V;
    for (uint32_t g = 0; g < v.G; ++g) {
        uint64_t *rec = v.pens + ((size_t)row * v.G + g) * v.pen_stride;
        const uint64_t h = rec[0];
        if (!(h & kPenDeferred))
            for (uint32_t i = (uint32_t)tid; i < (uint32_t)h; i += kThreads) {
                const uint64_t e = rec[1 + i];
                pen[(uint32_t)e] = __uint_as_float((uint32_t)(e >> 32));
            }
    }
    __syncthreads();
    if ((uint32_t)tid < v.G) v.pens[((size_t)row * v.G + tid) * v.pen_stride] = kPenDeferred;
    wait_vmem();
    __syncthreads();
}

// The sampled token's penalty: fma(old, decay, old == 0 ? presence : repetition) (reference:
// sampling.cu:427-437), the old value from the slice's notes (+0.0 when it is not among them).  A deferred
// slice still holds its old penalties and is rewritten whole by the fix-up kernel.
__device__ __forceinline__ void pen_patch(const Params &p, const StreamView &v, Lds &s, const uint32_t row, const uint32_t idx, const uint32_t slice_log2)
{
    const int tid = threadIdx.x;
    const uint64_t *rec = v.pens + ((size_t)row * v.G + (idx >> slice_log2)) * v.pen_stride;
    const uint64_t h = rec[0];
    if (h & kPenDeferred) return;
    if (tid == 0) s.bc32[6] = 0u;
    __syncthreads();
    for (uint32_t i = (uint32_t)tid; i < (uint32_t)h; i += kThreads) {
        const uint64_t e = rec[1 + i];
        if ((uint32_t)e == idx) s.bc32[6] = (uint32_t)(e >> 32);
    }
    __syncthreads();
    if (tid == 0) {
        const float old = __uint_as_float(s.bc32[6]);
        p.penalties[(int64_t)row * p.V + idx] = __builtin_fmaf(old, p.decay, old == 0.0f ? p.presence : p.repetition);
    }
}

// The last step of a pick: the token among at most 64 (index, weight) entries, in any order, at which the
// running sum of weights in index order reaches r.  One wave; lane i holds entry i, rank = the number of
// entries with a smaller index.  The entries go through LDS into index order, one scan does the rest.
__device__ __forceinline__ void pick_of_wave(const Params &p, LdsB &t, const uint32_t row, const int lane, const uint32_t n, const uint32_t rank,
                                             const uint32_t idx, const uint64_t w, const M96 r)
{
    if ((uint32_t)lane < n) { t.small[rank] = w; t.take[rank] = idx; }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const uint64_t wr = (uint32_t)lane < n ? t.small[lane] : 0ull;
    const uint32_t ir = t.take[lane];
    const Limbs mine = limbs(M96{wr, 0u}), upto = wave_inclusive_scan(mine);
    const M96 inc = m96(upto), exc = m96(upto - mine);
    if (exc < r && inc >= r) {
        p.out[row] = (int32_t)ir;
        if (p.diag) p.diag[row].index = (int32_t)ir;
        t.result = ir + 1u;
    }
}

// Finishes a row from what its slices published.  Returns true when the row is done (token written),
// false when it cannot be finished from the stashes: only on the one-launch path (FUSED = true: the
// caller is the last workgroup of the row to publish, the data was written by workgroups of this same
// launch and is read with device-scope atomic loads), where the caller then tells the row's other
// workgroups and the row's histogram is left in place for them.  With FUSED = false such a row is
// done here the slow way, from the logits, by the first four waves (the others have left: NT = 1024).
//
// What bounds it: nothing but the length of its chain.  A finish touches a few KB, and every step waits for
// the one before: trips to memory, scans, threshold, pick, with a workgroup barrier between most of them.
//   * The first 64 stashed tokens of every slice are asked for together with the headers and the row's
//     bins, before it is known which of them count: for the usual call that is all of them.  That nothing is
//     missing is checked by counting: the row's bins say how many tokens lie at or above the boundary bin.  A list
//     that may hold more takes the rest of each stash's prefix, as long as the slice's counts by bin say; those counts
//     are on their way while the first tokens are listed.  (Going through the stashes whole instead: 128 rows of 32768 with
//     top_k 1000 31.5 us a call against 21.7, one row of 524288 in 128 slices with top_k 50 24.4 against 14.5,
//     8 rows of 50304 with penalties and top_k 1000, in one launch, 28.6 against 19.5.)
//   * With one wave per SIMD (NT = 256) every wave works the one-wave steps out for itself: no barrier and no
//     trip through LDS for what all of them hold.
//   * The row's random number is drawn by a wave of its own (NT = 256: a fifth one, which leaves at its second
//     barrier; NT = 1024: the last; FUSED: drawn by the caller while its slice was on its way).
//   * Threshold and pick of a list of at most 64 tokens are one all-pairs step and one scan, wherever the list
//     comes from.  (Short lists out of whole stashes by digits and buckets: 1024 flat rows of 4096 with top_k 1 30.2 us a call
//     against 23.3, 288 of 8192 18.7 against 14.9.)
//   * Sums over a wave that need no carries (Limbs), no branch per list entry.
// Measured (cycles of 2.4 GHz in the workgroup, before: counts per slice fetched first, one wave for the scans with
// 128-bit sums, digits and buckets for every list): 13 rows of 50260, top_k 40: 14300 -> 9200; the kernel 7.6 -> 5.2 us;
// 256 rows of 151936: 9.2 -> 5.8 us; one row of 262144 with top_p 0.3: 8.0 -> 7.3.  Where they go now: the first trip to memory 2000,
// the level-1 scan 1800 (400 instructions), the list 1200, all pairs 650, threshold and target 1500, the pick 860.
// PRE: slices per wave whose first tokens are asked for ahead (W * PRE >= G for the short way).
// list: room for v.list_cap tokens in LDS.
template <int NT, int PRE, bool FUSED>
__device__ __forceinline__ bool finish_row(const Params &p, const StreamView &v, Lds &s, LdsB &t, uint64_t *list, const uint32_t row, const uint64_t drawn = 0)
{
    constexpr int  W = NT / kWave;
    constexpr bool kEach = NT == kThreads;               // every wave for itself
    static_assert(NT == 256 || NT == 1024, "one or four waves per SIMD");
    // the tokens asked for ahead may be listed a second time (FUSED with PRE = 16 never would, its list holds 2048 tokens, and has
    // no registers to keep them in)
    constexpr bool kAgain = !(FUSED && PRE > 8);
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = (int)uniform((uint32_t)tid >> 6);
    const uint32_t G = v.G;
    const PartHdr *hdrs = v.hdr + (size_t)row * G;
    const uint64_t *stash = v.stash + (size_t)row * G * kStashCap;
    uint64_t *rowhist = FUSED ? (p.ctl_end - 1 - row)->h[0] : (p.ctl_end - 1 - row)->rowhist;

    uint32_t rs[6] = {0u, 0u, 0u, 0u, 0u, 0u};
    uint32_t *rng_st = p.rng + (size_t)row * 16;
    const bool draws = !FUSED && wave == (kEach ? W : W - 1);
    if (draws && !p.inj_u) {
#pragma unroll
        for (int i = 0; i < 6; ++i) rs[i] = rng_st[i];
    }
    auto draw = [&]() {                                  // a row is always finished here unless FUSED: the state is advanced at once
        if (!p.inj_u) {
            uint32_t o[4];
            philox4x32_10(rs[2], rs[3], rs[4], rs[5], rs[0], rs[1], o);
            if (lane == 0) {
                t.rand64 = ((uint64_t)o[0] << 32) | o[1];
                rng_st[2] = rs[2] + 1u;
                if (rs[2] + 1u == 0u) rng_st[3] = rs[3] + 1u;
            }
        }
    };
    if (!FUSED && kEach && wave == W) {
        __syncthreads();
        draw();
        __syncthreads();
        return true;
    }
    PartHdr ph;
    ph.mkey = 0; ph.window = 0; ph.n = 0; ph.cut = 0;
    if ((uint32_t)tid < G) {
        if (FUSED) {
            const uint64_t *h2 = reinterpret_cast<const uint64_t *>(&hdrs[tid]);
            const uint64_t w0 = a_load(&h2[0]), w1 = a_load(&h2[1]);
            ph.mkey = (uint32_t)w0; ph.n = (uint32_t)w1; ph.cut = (uint32_t)(w1 >> 32);
        } else ph = hdrs[tid];
    }
    uint64_t h0 = 0, h1 = 0;
    if (kEach || tid < kThreads) { h0 = get<FUSED>(&rowhist[tid]); h1 = get<FUSED>(&rowhist[tid + kThreads]); }
    uint64_t pre[PRE];                                   // (slices beyond the row's read its last slice again and are set aside below)
#pragma unroll
    for (int i = 0; i < PRE; ++i) pre[i] = get<FUSED>(&stash[(size_t)min((uint32_t)(wave + W * i), G - 1u) * kStashCap + lane]);
    uint64_t *bk_lo = kEach ? t.blo : s.hr, *bk_hi = kEach ? t.bhi : s.hr + NT;       // buckets of the pick: NT of them
    static_assert(kEach || sizeof(s.hr) >= 2 * NT * sizeof(uint64_t), "room for the buckets");
    if (tid == 0) { s.abort = 0; s.host_words = p.host_words; t.result = 0u; s.ctr = 0u; t.nsmall = 0u; }
    if (FUSED && tid == kWave) t.rand64 = drawn;
    if (tid < 384) s.hm[tid] = 0;
    if (kEach && tid < 128) s.hm[256 + tid] = 0;
    bk_lo[tid] = 0; bk_hi[tid] = 0;

    // The headers and the row's bins into LDS, the row's frame from the slices' maxima.  Bins are read where they
    // lie, by absolute octave: bin r of the row's frame (octave M - 40 + r/4) sits at position 4 (M mod 128) + r - 160;
    // the 348 positions no bin of that frame falls on hold tokens below 2^-40, which are dead there.
    uint2 *hd = reinterpret_cast<uint2 *>(s.cand);       // per slice: key of its maximum, length of its stash
    static_assert(sizeof(s.cand) >= kMaxParts * sizeof(uint2), "the headers lie in s.cand");
    uint32_t kmax, kmin;
    {
        const uint32_t a = wave_max_u32(ph.mkey), b = wave_max_u32((uint32_t)tid < G ? ~ph.mkey : 0u);
        if (lane == 0) { t.take[wave] = a; t.take[W + wave] = b; }
        if (tid < kMaxParts) hd[tid] = make_uint2(ph.mkey, min(ph.n, (uint32_t)kStashCap));
        if (kEach || tid < kThreads) {
            s.g[tid] = h0; s.g[tid + kThreads] = h1;
            if (!FUSED) { rowhist[tid] = 0; rowhist[tid + kThreads] = 0; }               // left clean for the next call
        }
        __syncthreads();
        kmax = t.take[0]; kmin = t.take[W];
        constexpr int kHdrWaves = kEach ? W : kMaxParts / kWave;       // the waves that hold headers
#pragma unroll
        for (int w = 1; w < kHdrWaves; ++w) { kmax = max(kmax, t.take[w]); kmin = max(kmin, t.take[W + w]); }
        kmax = uniform(kmax); kmin = ~uniform(kmin);
    }
    if (!kEach && draws) draw();
    const float xmax = fkey_inv(kmax);
    const float M = __builtin_floorf(xmax);
    // frames further apart than this may have put different octaves into one bin
    const bool mixed = !(M - __builtin_floorf(fkey_inv(kmin)) < 88.0f);
    const float mm = M - 128.0f * __builtin_floorf(M * 0.0078125f);
    const uint32_t m4 = (uint32_t)(int)mm * 4u;
    auto octaves_below = [&](uint32_t key) {             // of a slice's frame below the row's, at most 64
        const float d = M - __builtin_floorf(fkey_inv(key));          // >= 0, a whole number or huge
        return d >= 64.0f ? 64u : (uint32_t)d;
    };
    auto pos = [&](uint32_t b) { return (m4 + b - kBin0 - 160u) & 511u; };       // position of level-1 bin b
    if (__builtin_expect(mixed, 0)) {
        // Slices whose maxima lie 88 octaves or more apart may have put different octaves into
        // one position.  Every token of a slice 41 octaves or more below the row's frame is
        // dead there, whatever its bin: what such a slice added is taken out again, bin by bin
        // (its own bins are on record).  The slices that remain lie within 40 octaves of each
        // other.
        for (uint32_t i = (uint32_t)tid; i < G * (uint32_t)kSB; i += NT) {
            const uint32_t g = i / (uint32_t)kSB, r = i - g * (uint32_t)kSB;
            if (octaves_below(hd[g].x) >= 41u) {
                const uint64_t w = get<FUSED>(&v.shist[((size_t)row * G + g) * kSB + r]);
                if (w) {
                    const float Mg = __builtin_floorf(fkey_inv(hd[g].x));
                    const uint32_t mg4 = (uint32_t)(int)(Mg - 128.0f * __builtin_floorf(Mg * 0.0078125f)) * 4u;
                    atomicAdd(reinterpret_cast<unsigned long long *>(&s.g[(mg4 + r - 160u) & 511u]), 0ull - (unsigned long long)w);
                }
            }
        }
        __syncthreads();
    }
    if (__builtin_expect(p.e_bits != nullptr, 0)) {
        // diagnostics: the slices' e into the row's frame, dead tokens as 0
        uint4 *eb4 = reinterpret_cast<uint4 *>(p.e_bits + (int64_t)row * p.V);
        auto fix = [&](uint32_t b, uint32_t d) { b = rebase_bits(min(b, 0x3FFFFFFFu), d); return b < kEMinBits ? 0u : b; };
        for (uint32_t i4 = (uint32_t)tid; i4 < ((uint32_t)p.V >> 2); i4 += NT) {
            const uint32_t d = octaves_below(hd[i4 >> (v.slice_log2 - 2u)].x);
            uint4 q;
            if (FUSED) {
                const uint32_t *w = reinterpret_cast<const uint32_t *>(&eb4[i4]);
                q = make_uint4(a_load(&w[0]), a_load(&w[1]), a_load(&w[2]), a_load(&w[3]));
            } else q = eb4[i4];
            q.x = fix(q.x, d); q.y = fix(q.y, d); q.z = fix(q.z, d); q.w = fix(q.w, d);
            if (FUSED) {
                // written through: a workgroup that falls back rewrites its slice of this later
                uint32_t *w = reinterpret_cast<uint32_t *>(&eb4[i4]);
                a_store(&w[0], q.x); a_store(&w[1], q.y); a_store(&w[2], q.z); a_store(&w[3], q.w);
            } else eb4[i4] = q;
        }
    }

    // A step one wave does: the first wave's result by way of LDS, unless every wave does it for itself.
    struct { uint32_t place, cnt_above, cnt_bin; M96 above; } f;
    f.place = 0; f.cnt_above = 0; f.cnt_bin = 0; f.above = M96{0ull, 0u};
    M96 D{0ull, 0u}, P{0ull, 0u};
    auto hand_on = [&](bool found) -> bool {
        if constexpr (kEach) return found;
        if (tid == 0) {
            t.one.D = D; t.one.P = P; t.one.above = f.above;
            t.one.place = f.place; t.one.cnt_above = f.cnt_above; t.one.cnt_bin = f.cnt_bin; t.one.found = found ? 1u : 0u;
        }
        __syncthreads();
        D = uniform(t.one.D); P = uniform(t.one.P); f.above = uniform(t.one.above);
        f.place = uniform(t.one.place); f.cnt_above = uniform(t.one.cnt_above); f.cnt_bin = uniform(t.one.cnt_bin);
        return uniform(t.one.found) != 0u;
    };
    const uint32_t top_k = (uint32_t)p.top_k;
    // boundary bin of the row, with D and P (whole_row), or of the listed tokens alone (counted in s.g by bin)
    auto level1 = [&](bool whole_row) -> bool {
        bool found = false;
        if (kEach || wave == 0) {
            BinScan<3> sc;
            auto at = [&](int i) { return (uint32_t)max((int)kTop1 - 3 * lane - i, (int)kBin0); };
            auto live = [&](int i) { return (int)kTop1 - 3 * lane - i >= (int)kBin0; };
            sc.load([&](int i) { const uint64_t w = s.g[whole_row ? pos(at(i)) : at(i)]; return live(i) ? w : 0ull; }, [&](int i) { return at(i) >> 2; });
            if (whole_row) { D = sc.total(); P = ceil_mul(p.top_p, D); }
            found = sc.search(0u, M96{0ull, 0u}, top_k, P, f.place, f.cnt_above, f.cnt_bin, f.above);
        }
        return hand_on(found);
    };
    level1(true);
    uint32_t bin = kTop1 - f.place;

    // What the stashes cannot finish, this workgroup does alone from the logits.  Such rows are
    // counted, and the first of a call tells the caller's policy at once (that a call went well is
    // reported by the call after it, see report_begin).
    auto tell_policy = [&](const Params &p) {
        if (tid == 0) {
            const uint32_t c = __hip_atomic_fetch_add(&p.hdr->n_need, 1u, __ATOMIC_RELAXED, RS_AGENT);
            if (c == 0u && p.host_words)                 // the call's first such row tells the caller's policy at once
                __hip_atomic_store(p.host_words + p.report, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    };

    // A row that is one tie of all its tokens (rows of equal logits) needs no stash at all: the
    // threshold is the largest token's value, every token weighs the tie weight, and the token at
    // which the running sum reaches r follows by division.
    if (__builtin_expect(f.cnt_bin == (uint32_t)p.V, 0)) {
        const uint32_t emax = e_bits_of(xmax, M);
        if (bin_is_one_tie(uniform(s.g[pos(bin)]), bin, emax)) {
            __syncthreads();                             // the random number is there
            if (tid == 0) {
                const Target tg = tie_and_target(p, row, t.rand64, xmax, wide(D), wide(P), emax, 0u, f.cnt_bin, (u128)0, 0u, true);
                // smallest i with (i + 1) * w_tie >= r; r <= V * w_tie
                uint32_t lo_i = 0, hi_i = (uint32_t)p.V - 1u;
                while (lo_i < hi_i) {
                    const uint32_t mid = (lo_i + hi_i) >> 1;
                    if ((u128)(mid + 1u) * tg.w_tie >= tg.r) hi_i = mid; else lo_i = mid + 1u;
                }
                p.out[row] = (int32_t)lo_i;
                if (p.diag) p.diag[row].index = (int32_t)lo_i;
                t.result = lo_i + 1u;
            }
            return true;
        }
    }

    // ---- the list: the row's tokens at or above the boundary bin ----
    auto claim = [&](uint32_t n) {
        uint32_t at = 0;
        if (lane == 0 && n) at = atomicAdd(&s.ctr, n);
        return uniform(at);
    };
    const uint32_t total = f.cnt_above + f.cnt_bin;
    const uint32_t cut = bin << 21;
    uint32_t n = 0;                                      // tokens listed
    bool listed = false, subset = false;
    const bool ahead = total <= v.list_cap && G <= (uint32_t)(W * PRE);
    // How many tokens of slice tid lie at or above the boundary bin, as its workgroup counted them: asked for while the
    // first ones go into the list if those may well not be all (more than 40 a slice on average), else when they are not.
    auto octaves = [&]() { return (uint32_t)tid < G ? octaves_below(ph.mkey) : 0u; };
    auto count_above = [&]() -> uint32_t {
        const uint32_t lb = bin - kBin0 + 4u * octaves();   // the boundary bin in the slice's frame; past its last bin: nothing of the slice is live
        return (uint32_t)tid < G && lb < (uint32_t)kSB ? get<FUSED>(&v.cum[((size_t)row * G + (uint32_t)tid) * kSB + lb]) : 0u;
    };
    const bool likely = !ahead || total > max((uint32_t)kWave, 40u * G);
    uint32_t above_cut = 0;
    if (likely) {
        // (The first tokens have long arrived.  Said here, because behind a load that not every thread makes the compiler
        // waits for that load, too, before it touches them.)
        __builtin_amdgcn_s_waitcnt(0x0F70);              // vmcnt(0)
        above_cut = count_above();
    }
    // The tokens asked for ahead, those at or above `from` of them into the list.  Called by all threads together, s.ctr = 0.
    auto list_ahead = [&](const uint32_t from) -> uint32_t {
        // lane i looks after the wave's i-th slice: how far its frame lies below the row's, how many tokens it stashed
        const uint32_t sl = (uint32_t)(wave + W * lane);
        const uint2 h = hd[min(sl, G - 1u)];
        const uint32_t below = octaves_below(h.x), len = sl < G ? min(h.y, (uint32_t)kWave) : 0u;
        uint64_t e[PRE];
        uint32_t mine = 0;                               // of this lane's tokens, how many
#pragma unroll
        for (int i = 0; i < PRE; ++i) {
            const uint32_t b = rebase_bits((uint32_t)(pre[i] >> 32), lane_of(below, (uint32_t)i));
            const bool in = (uint32_t)lane < lane_of(len, (uint32_t)i) && b >= from;
            e[i] = ((uint64_t)(in ? b : 0u) << 32) | (uint32_t)pre[i];
            mine += in ? 1u : 0u;
        }
        const uint32_t upto = wave_inclusive_scan(mine);
        uint32_t at = claim(lane63(upto)) + upto - mine;
#pragma unroll
        for (int i = 0; i < PRE; ++i)
        {
            // (a branch per entry would cost more than the store: what is not listed goes into a corner of its own)
            typedef __attribute__((address_space(3))) uint64_t lds_u64;
            const bool in = (uint32_t)(e[i] >> 32) != 0u;
            lds_u64 *to = in ? (lds_u64 *)list + at : (lds_u64 *)t.small + lane;
            *to = e[i];
            at += in ? 1u : 0u;
        }
        __syncthreads();
        return uniform(s.ctr);
    };
    if (ahead) {
        n = list_ahead(cut);
        listed = n == total;                             // every token at or above the boundary bin is there
    }
    if (__builtin_expect(!listed, 0)) {                  // (out of the way of the usual call's instructions)
        // Prefixes of the stashes, one after the other: t.take[g] = entries of slices 0..g.  Returns how many in all.
        auto take_prefix = [&](uint32_t mine) -> uint32_t {
            uint32_t inc = wave_inclusive_scan(mine);
            __syncthreads();
            if (lane == kWave - 1) s.u32[wave] = inc;
            __syncthreads();
            uint32_t sum = 0;
#pragma unroll
            for (int w = 0; w < kMaxParts / kWave; ++w) {              // the waves that hold slices
                if (w < wave) inc += s.u32[w];
                sum += s.u32[w];
            }
            if (tid < kMaxParts) t.take[tid] = inc;
            __syncthreads();
            return uniform(sum);
        };
        // fn(i, step, bits of e in the row's frame, tokens) for the n_all entries t.take speaks of, those of a slice from entry
        // `skip` on: eight of a thread at a time and in flight together, entries i, i + step, ... (bits 0 past the last).  A
        // thread looks up the slice of its first entry and walks on from there.  Many entries per slice: neighbouring
        // threads read neighbouring entries (512 flat rows of 131072 with top_k 1000 104 us a call, 114 in runs); few: a thread reads a run of them, which
        // takes it over fewer slices (one row of 524288 in 128 slices with top_k 200: 15 us a call, 19.7 with neighbours).
        // Called by all threads together.
        constexpr int kBatch = 8;
        auto stashed = [&](const uint32_t n_all, const uint32_t skip, auto fn) {
            const uint32_t per = (n_all + (uint32_t)NT - 1u) / (uint32_t)NT;
            const bool dense = n_all >= 64u * G;
            const uint32_t first = dense ? (uint32_t)tid : (uint32_t)tid * per, step = dense ? (uint32_t)NT : 1u;
            uint32_t g = 0, hi_g = G - 1u;                             // first slice whose prefix exceeds the first entry
            while (g < hi_g) {
                const uint32_t mid = (g + hi_g) >> 1;
                if (t.take[mid] > first) hi_g = mid; else g = mid + 1u;
            }
            uint32_t gend = t.take[g];
            const uint64_t *from_g = stash + (size_t)g * kStashCap + skip - (g ? t.take[g - 1u] : 0u);
            for (uint32_t k = 0; k < per; k += (uint32_t)kBatch) {
                uint64_t e[kBatch];
                uint32_t d[kBatch];
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    const uint32_t i = first + (k + (uint32_t)u) * step;
                    e[u] = 0; d[u] = 0;
                    if (k + (uint32_t)u < per && i < n_all) {
                        while (i >= gend) {                            // slices that give nothing are skipped
                            ++g; from_g = stash + (size_t)g * kStashCap + skip - gend; gend = t.take[g];
                        }
                        e[u] = get<FUSED>(&from_g[i]);
                        d[u] = t.delta[g];
                    }
                }
                uint32_t bits[kBatch], idx[kBatch];
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    bits[u] = (uint32_t)(e[u] >> 32) ? rebase_bits((uint32_t)(e[u] >> 32), d[u]) : 0u;
                    idx[u] = (uint32_t)e[u];
                }
                fn(first + k * step, step, bits, idx);
            }
        };
        // the tokens at or above `from` among them, side by side
        auto list_from = [&](const uint32_t n_all, const uint32_t from) -> uint32_t {
            __syncthreads();                             // the list's counter has been read
            if (tid == 0) s.ctr = 0u;
            __syncthreads();
            stashed(n_all, 0u, [&](uint32_t, uint32_t, const uint32_t (&bits)[kBatch], const uint32_t (&idx)[kBatch]) {
                uint32_t mine = 0;
#pragma unroll
                for (int u = 0; u < kBatch; ++u) mine += bits[u] >= from ? 1u : 0u;
                const uint32_t upto = wave_inclusive_scan(mine);
                uint32_t at = claim(lane63(upto)) + upto - mine;
#pragma unroll
                for (int u = 0; u < kBatch; ++u)
                    if (bits[u] >= from) {
                        if (at < v.list_cap) list[at] = ((uint64_t)bits[u] << 32) | idx[u];
                        ++at;
                    }
            });
            __syncthreads();
            return uniform(s.ctr);
        };
        const uint32_t dl = octaves();
        if ((uint32_t)tid < G) t.delta[tid] = dl;
        if (!likely) above_cut = count_above();
        // Together the stashes hold every token of the row at or above `from`, the largest of the slices' cuts.  (A
        // cut that lands below 2^-40 in the row's frame: what the stash lacks is dead there.)
        const uint32_t len = (uint32_t)tid < G ? min(ph.n, (uint32_t)kStashCap) : 0u;
        uint32_t from = (uint32_t)tid < G ? max(rebase_bits(ph.cut, dl), kEMinBits) : 0u;
        from = wave_max_u32(from);
        uint32_t longer = __builtin_amdgcn_ballot_w64(len > (uint32_t)kWave) != 0ull ? 1u : 0u;        // some stash than what was asked for ahead
        __syncthreads();
        if (lane == 0) { t.take[wave] = from; t.take[W + wave] = longer; }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kMaxParts / kWave; ++w) { from = max(from, t.take[w]); longer |= t.take[W + w]; }
        from = uniform(from); longer = uniform(longer);
        bool slow = false;
        uint32_t list_all = 0;                           // stashed tokens to go through for those at or above `from`
        if (from <= cut && total <= v.list_cap) {        // plan A: every stash reaches down to the boundary bin
            // exactly the tokens at or above that bin: of every stash a prefix, whose first 64 are listed already
            const uint32_t skip = ahead ? (uint32_t)kWave : 0u, had = n, take = min(above_cut, len);
            const uint32_t rest = take_prefix(take > skip ? take - skip : 0u);
            n = had + rest;
            slow = n != total;
            if (!slow)
                stashed(rest, skip, [&](uint32_t i, uint32_t step, const uint32_t (&bits)[kBatch], const uint32_t (&idx)[kBatch]) {
#pragma unroll
                    for (int u = 0; u < kBatch; ++u)
                        if (bits[u]) list[had + i + (uint32_t)u * step] = ((uint64_t)bits[u] << 32) | idx[u];
                });
            __syncthreads();
        } else if (kAgain && !longer && G <= (uint32_t)(W * PRE) && G * (uint32_t)kWave <= v.list_cap) {
            // plan B, the stashes whole, every one of them asked for ahead (320 flat rows of 8192 with penalties, top_k 50:
            // 23.2 us a call from the stashes again, 22.6 this way)
            if (tid == 0) s.ctr = 0u;                    // (it has been read)
            __syncthreads();
            n = list_ahead(from);
            subset = true;
        } else if (const uint32_t all = take_prefix(len); !FUSED && all > min(v.list_cap, max(2048u, 3u * top_k)) && top_k <= v.list_cap / 2u) {
            // Plan B (flat distributions: the boundary bin holds thousands of tokens, but top_k is small) with more
            // stashed tokens than the list holds, or several times top_k of them.  The kept set is at most
            // top_k tokens, so only the stashed tokens down to some value T at or above which there are at least
            // top_k of them are needed: T from a count of the stashed tokens in steps of 1/512 octave below the
            // row's largest (one pass over the stashes, which sit in the L2), the tokens at or above T into the
            // list by a second pass.  T is at or above `from`, so the list is complete above T.
            const uint32_t topkey = e_bits_of(xmax, M) >> 14;
            uint32_t *cnt = reinterpret_cast<uint32_t *>(s.cand);                // 512 counters
            if (tid < 512) cnt[tid] = 0u;
            if (kEach) cnt[256 + tid] = 0u;
            if (tid == 0) { s.bc32[4] = 0xFFFFFFFFu; s.bc32[5] = 0u; }
            __syncthreads();
            stashed(all, 0u, [&](uint32_t, uint32_t, const uint32_t (&bits)[kBatch], const uint32_t (&)[kBatch]) {
#pragma unroll
                for (int u = 0; u < kBatch; ++u)
                    if (bits[u] >= from) atomicAdd(&cnt[min(511u, topkey - (bits[u] >> 14))], 1u);
            });
            __syncthreads();
            if (wave == 0) {
                uint32_t c8 = 0;
#pragma unroll
                for (int q = 0; q < 8; ++q) c8 += cnt[lane * 8 + q];
                const uint32_t inc = wave_inclusive_scan(c8);
                uint32_t run = inc - c8;
                if (run < top_k && top_k <= inc) {
                    bool done = false;
#pragma unroll
                    for (int q = 0; q < 8; ++q) {
                        run += cnt[lane * 8 + q];
                        if (!done && run >= top_k) { s.bc32[4] = (uint32_t)(lane * 8 + q); s.bc32[5] = run; done = true; }
                    }
                }
            }
            __syncthreads();
            const uint32_t step = uniform(s.bc32[4]), nge = uniform(s.bc32[5]);
            slow = step >= 511u || nge > v.list_cap;     // fewer than top_k at or above `from`, or one value thousands of times
            if (!slow) {
                list_all = all;
                from = max(from, (topkey - step) << 14);
                // Two more passes over the stashes make this finish slower than the general kernel's whole
                // call while the call is of moderate size (measured: 64 flat rows of 131072 with top_k 1000,
                // 44 against 38 us; 128 rows of 262144, 68 against 116): such a call says so to the caller's
                // policy, as it did when these rows still went the slow way.
                // (p.tell_lists: calls of fewer than 2^24 tokens, and calls whose rows the row kernel would take)
                if (p.tell_lists) tell_policy(params_again());
            }
        } else {                                         // plan B, the stashes whole
            slow = all > v.list_cap || all == 0u;
            if (!slow) list_all = all;
        }
        if (list_all) { n = list_from(list_all, from); subset = true; }
        // A short list of at least top_k tokens holds the kept set; of any other it is the listed tokens' own bins that say
        // whether it does.
        if (!slow && subset && (n < top_k || n > (uint32_t)kWave)) {
            // level 1 again, on the listed tokens alone
            __syncthreads();
            for (int b = tid; b < kSB; b += NT) s.g[kBin0 + b] = 0;
            __syncthreads();
            for (uint32_t i = (uint32_t)tid; i < n; i += NT) {
                const uint32_t b = (uint32_t)(list[i] >> 32);
                atomicAdd(reinterpret_cast<unsigned long long *>(&s.g[b >> 21]), (unsigned long long)(kPackOne | (b & 0x7FFFFFu)));
            }
            __syncthreads();
            slow = !level1(false);                       // even all of them are neither top_k tokens nor top_p of the mass
            bin = kTop1 - f.place;
        }
        if (slow) {
            if (FUSED) return false;
            __syncthreads();                             // the random number is there
            if (NT > kThreads && tid >= kThreads) return true;
            const Params q = params_again();
            if (q.penalties && q.defer_pen == 2) pen_restore(q, v, row);
            finish_row_slow(q, s, t, row, xmax, q.inj_u ? 0ull : t.rand64);
            tell_policy(q);
            return true;
        }
    }

    // a list so long that another kernel is faster (the host's rule): said to the caller's policy
    if (!FUSED && n > p.long_list) tell_policy(params_again());

    if (n <= (uint32_t)kWave) {
        // ---- a short list: every pair of its tokens ----
        // Lane i of each of four waves holds token i and goes through a quarter of the others: how many are larger,
        // what they weigh, how many come before it in index order.  A token is kept when what is larger is neither
        // top_k tokens nor P; the threshold is the smallest kept value.
        struct Part { uint64_t lo; uint32_t hi, cnt; };              // cnt: larger | before << 16
        Part *part = reinterpret_cast<Part *>(s.cand);               // [4][64]
        static_assert(sizeof(Part) == 16 && sizeof(s.cand) >= 4 * kWave * sizeof(Part) && offsetof(Lds, cand) % 16 == 0, "partial sums live in s.cand");
        const uint64_t e = list[min((uint32_t)lane, n - 1u)];
        const uint32_t b = (uint32_t)(e >> 32), idx = (uint32_t)e;
        if (wave < 4) {
            M96 sum{0ull, 0u};
            uint32_t larger = 0, before = 0;
            const uint32_t per = (n + 3u) >> 2, j1 = min(n, ((uint32_t)wave + 1u) * per);
#pragma unroll 4
            for (uint32_t j = (uint32_t)wave * per; j < j1; ++j) {
                const uint64_t o = list[j];
                const bool gt = (uint32_t)(o >> 32) > b;
                sum = sum + M96{gt ? w_of_bits((uint32_t)(o >> 32)) : 0ull, 0u};
                larger += gt ? 1u : 0u;
                before += (uint32_t)o < idx ? 1u : 0u;
            }
            part[wave * kWave + lane] = Part{sum.lo, sum.hi, larger | before << 16};
        }
        __syncthreads();
        if (wave == 0) {
            M96 above{0ull, 0u};
            uint32_t cnt = 0;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const Part q = part[w * kWave + lane];
                above = above + M96{q.lo, q.hi};
                cnt += q.cnt;
            }
            const uint32_t larger = cnt & 0xFFFFu, rank = cnt >> 16;
            const bool in = (uint32_t)lane < n;
            const bool kept = in && larger < top_k && above < P;
            const uint32_t thr = ~wave_max_u32(kept ? ~b : 0u);
            const uint64_t ties = __builtin_amdgcn_ballot_w64(in && b == thr);
            const uint32_t l = (uint32_t)__builtin_ctzll(ties);
            const Target tg = tie_and_target(p, row, t.rand64, xmax, wide(D), wide(P), thr, lane_of(larger, l), (uint32_t)__builtin_popcountll(ties),
                                             wide(lane_of(above, l)), 0u, lane == 0);            // rounds = 0: no cluster histogram
            pick_of_wave(p, t, row, lane, n, rank, idx, b > thr ? w_of_bits(b) : b == thr ? tg.w_tie : 0ull, m96(tg.r));
        }
        return true;
    }

    // ---- a longer list: the remaining digits of the threshold ----
    uint32_t lo = bin << 21, span = (1u << 21) - 1u;
    const uint32_t exb = bin >> 2;
    for (uint32_t lv = 2; lv <= (uint32_t)kLevels && f.cnt_bin > 1u; ++lv) {
        const uint32_t dsh = level_shift(lv);
        uint64_t *hist = s.hm + (lv - 2u) * 128u;
        for (uint32_t i = (uint32_t)tid; i < n; i += NT) {
            const uint32_t b = (uint32_t)(list[i] >> 32);
            if (b - lo <= span) atomicAdd(reinterpret_cast<unsigned long long *>(&hist[(b >> dsh) & 127u]), (unsigned long long)(kPackOne | (b & 0x7FFFFFu)));
        }
        __syncthreads();
        bool found = true;
        if (kEach || wave == 0) {
            BinScan<2> sc;
            sc.load([&](int i) { return hist[127 - 2 * lane - i]; }, [&](int) { return exb; });
            const uint32_t c0 = f.cnt_above;
            const M96 m0 = f.above;
            found = sc.search(c0, m0, top_k, P, f.place, f.cnt_above, f.cnt_bin, f.above);
        }
        hand_on(found);
        lo |= (127u - f.place) << dsh;
        span = (1u << dsh) - 1u;
    }
    if (span != 0u) {                                    // a single token left in the range: the threshold itself
        for (uint32_t i = (uint32_t)tid; i < n; i += NT) {
            const uint32_t b = (uint32_t)(list[i] >> 32);
            if (b - lo <= span) s.bc32[6] = b;
        }
        __syncthreads();
        lo = uniform(s.bc32[6]);
    }
    const uint32_t thr = lo;
    uint64_t w_tie = 0;
    M96 r{0ull, 0u};
    if (kEach || wave == 0) {
        const Target tg = tie_and_target(p, row, t.rand64, xmax, wide(D), wide(P), thr, f.cnt_above, f.cnt_bin, wide(f.above), 0u, tid == 0);
        w_tie = tg.w_tie; r = m96(tg.r);
    }
    if constexpr (!kEach) {
        if (tid == 0) { s.bc64[1] = w_tie; t.one.P = r; }
        __syncthreads();
        w_tie = uniform(s.bc64[1]); r = uniform(t.one.P);
    }

    // ---- the pick: kept weights by bucket of the token index, NT buckets a step, then the bucket's tokens ----
    // (a weight is below 2^64 and a bucket has fewer than 2^14 listed tokens: the halves summed apart stay below 2^46)
    auto weight = [=](uint32_t b) -> uint64_t { return (b > thr) ? w_of_bits(b) : (b == thr ? w_tie : 0ull); };
    constexpr uint32_t kLogNT = NT == 256 ? 8u : 10u;
    uint32_t sh = 32u - (uint32_t)__builtin_clz((uint32_t)p.V - 1u | 1u);
    sh = sh > kLogNT ? sh - kLogNT : 0u;
    uint32_t lo_idx = 0, len = (uint32_t)p.V;
    // (kept tokens few enough for one wave as they are: no buckets.  320 flat rows of 8192 with penalties, top_k 50: 23.6 -> 23.2 us a call)
    bool few = f.cnt_above + f.cnt_bin <= (uint32_t)kWave;
    uint32_t *ranks = reinterpret_cast<uint32_t *>(s.cand + kWave);    // [4][64]
    static_assert(sizeof(s.cand) >= 3 * kWave * sizeof(uint64_t), "the ranks lie behind the tokens in s.cand");
    for (;; few = false) {
        if (!few) {
            for (uint32_t i = (uint32_t)tid; i < n; i += NT) {
                const uint64_t e = list[i];
                const uint32_t off = (uint32_t)e - lo_idx;
                const uint64_t w = weight((uint32_t)(e >> 32));
                if (w && off < len) {
                    atomicAdd(reinterpret_cast<unsigned long long *>(&bk_lo[off >> sh]), (unsigned long long)(w & 0xFFFFFFFFull));
                    atomicAdd(reinterpret_cast<unsigned long long *>(&bk_hi[off >> sh]), (unsigned long long)(w >> 32));
                }
            }
            __syncthreads();
            const M96 mine = m96((u128)bk_lo[tid] + ((u128)bk_hi[tid] << 32));
            bk_lo[tid] = 0; bk_hi[tid] = 0;
            M96 inc = m96(wave_inclusive_scan(limbs(mine)));
            M96 *waves = reinterpret_cast<M96 *>(&s.wj[0][0]);
            static_assert(sizeof(s.wj) >= 16 * sizeof(M96), "one mass per wave");
            if (lane == kWave - 1) waves[wave] = inc;
            __syncthreads();
            {
                const Limbs tot = wave_inclusive_scan(limbs(lane < W ? waves[lane] : M96{0ull, 0u}));
                if (wave) inc = inc + m96(lane_of(tot, (uint32_t)wave - 1u));
            }
            const M96 exc = inc - mine;
            if (exc < r && inc >= r) { t.bucket = (uint32_t)tid; t.one.above = r - exc; }
            __syncthreads();
            lo_idx += uniform(t.bucket) << sh; len = 1u << sh;
            r = uniform(t.one.above);
        }
        // the kept tokens of the bucket: few enough for one wave, as a rule; otherwise the bucket is cut into NT again
        for (uint32_t i = (uint32_t)tid; i < n; i += NT) {
            const uint64_t e = list[i];
            if ((uint32_t)e - lo_idx < len && weight((uint32_t)(e >> 32))) {
                const uint32_t o = atomicAdd(&t.nsmall, 1u);
                if (o < (uint32_t)kWave) s.cand[o] = e;
            }
        }
        __syncthreads();
        const uint32_t ns = uniform(t.nsmall);
        if (ns <= (uint32_t)kWave) {
            // how many of them come before each: one wave alone or, of more than a few, four with a quarter each
            const uint64_t e = s.cand[min((uint32_t)lane, ns - 1u)];
            const bool split = ns > 16u;
            const uint32_t per = split ? (ns + 3u) >> 2 : ns, j1 = min(ns, ((uint32_t)wave + 1u) * per);
            uint32_t rank = 0;
#pragma unroll 4
            for (uint32_t j = (uint32_t)wave * per; j < j1; ++j) rank += (uint32_t)s.cand[j] < (uint32_t)e ? 1u : 0u;
            if (split) {
                if (wave < 4) ranks[wave * kWave + lane] = rank;
                __syncthreads();
                rank = ranks[lane] + ranks[kWave + lane] + ranks[2 * kWave + lane] + ranks[3 * kWave + lane];
            }
            if (wave == 0) {
                pick_of_wave(p, t, row, lane, ns, rank, (uint32_t)e, weight((uint32_t)(e >> 32)), r);
            }
            return true;
        }
        __syncthreads();                                 // everyone has read the count
        if (tid == 0) t.nsmall = 0u;
        sh = sh > kLogNT ? sh - kLogNT : 0u;
        __syncthreads();
    }
}

// NT: 256 threads and the wave that draws the random number, or 1024 for calls whose lists are long (the host's choice).
template <int NT> constexpr int finish_threads() { return NT == kThreads ? NT + kWave : NT; }
template <int NT, int PRE>
__global__ void __launch_bounds__(finish_threads<NT>()) finish_kernel(const Params p, const StreamView v)
{
    __shared__ Lds s;
    __shared__ LdsB t;
    extern __shared__ __align__(16) unsigned char finish_dyn[];
    finish_row<NT, PRE, false>(p, v, s, t, reinterpret_cast<uint64_t *>(finish_dyn), blockIdx.x);
    if (p.penalties && p.defer_pen == 2) {
        if (threadIdx.x >= kThreads) return;
        __syncthreads();
        pen_patch(p, v, s, blockIdx.x, t.result - 1u, v.slice_log2);
    }
}

// ---- calls that keep every live token (top_k = V, top_p = 1): one workgroup per row behind the counting-only pass ----
// The pass left, per slice, its mass without its lowest 4 d bins for every d (41 sums): a slice whose frame lies d
// octaves below the row's has just those bins dead in the row's frame, and what is left is a multiple of 2^d.  So
// the row's total and the slice that holds the target come from one load and one scan per wave -- every wave does
// them for itself -- and only that slice's logits are looked at again.
//
// What bounds it: the length of the chain (headers -> target -> slice -> token), two trips to memory of a
// microsecond each.  The slice comes in coalesced and goes through LDS, so that every thread then owns consecutive
// tokens: one sum per thread, one scan over the workgroup, and one wave finds the token among the owner's T.
// (Chunks of 256 consecutive tokens summed wave by wave, two 64-bit wave sums each, behind the general finish's bins and
// boundary: 16.1 us for 512 rows of 50304 tokens; this way 10.8, of which some 5 are the 16 MB of slices.)
constexpr int kKeepT = 512;                              // threads that look at the slice; one more wave draws the random number
template <int LOG2>
struct LdsK {
    static constexpr int U = (1 << LOG2) / 4 / kKeepT;   // float4 groups per thread
    float4   x[kKeepT * U + kKeepT];                     // group g of the slice at g + g / U: threads read their U groups an odd number of groups apart
    M96      waves[kKeepT / kWave];
    uint64_t rand64;
    uint32_t u32[kKeepT / kWave];
};

// The diagnostics record of such a call names the threshold -- the smallest live token of the row -- and how many
// tokens tie there: one pass over the row, paid by callers that ask for the record (tests, mostly).
template <typename L>
__device__ __forceinline__ void keep_diag(const Params &p, L &s, const uint32_t row, const float xmax, const M96 D, const uint64_t rand64)
{
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    const float M = __builtin_floorf(xmax);
    const char *lrow = logits_row(p, row);
    auto each = [&](auto fn) {
        for (uint32_t i4 = (uint32_t)tid; i4 < (uint32_t)p.V >> 2; i4 += kKeepT) {
            const float4 l = load_logits4(lrow, i4, p.dtype);
            fn(e_bits_of(sf(l.x * p.c), M)); fn(e_bits_of(sf(l.y * p.c), M)); fn(e_bits_of(sf(l.z * p.c), M)); fn(e_bits_of(sf(l.w * p.c), M));
        }
    };
    auto over_waves = [&](uint32_t v, bool sum) {        // sum or minimum over the workgroup
        v = sum ? wave_sum(v) : ~wave_max_u32(~v);
        __syncthreads();
        if (lane == 0) s.u32[wave] = v;
        __syncthreads();
        uint32_t r = s.u32[0];
        for (int w = 1; w < kKeepT / kWave; ++w) r = sum ? r + s.u32[w] : min(r, s.u32[w]);
        return r;
    };
    uint32_t mn = 0xFFFFFFFFu, n_live = 0, n_eq = 0;
    each([&](uint32_t b) { if (b >= kEMinBits) { mn = min(mn, b); ++n_live; } });
    mn = over_waves(mn, false);
    each([&](uint32_t b) { if (b == mn) ++n_eq; });
    n_live = over_waves(n_live, true); n_eq = over_waves(n_eq, true);
    if (tid == 0)
        tie_and_target(p, row, rand64, xmax, wide(D), wide(D), mn, n_live - n_eq, n_eq, wide(D) - (u128)n_eq * w_of_bits(mn), 9u, true);
}

template <int LOG2>
__global__ void __launch_bounds__(kKeepT + kWave) keep_finish_kernel(const Params p, const StreamView v)
{
    __shared__ LdsK<LOG2> s;
    constexpr int U = LdsK<LOG2>::U, T = 4 * U;          // groups and tokens per thread
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = (int)uniform((uint32_t)tid >> 6);
    const uint32_t row = blockIdx.x, G = v.G, V4 = (uint32_t)p.V >> 2;
    if (wave == kKeepT / kWave) {
        if (!p.inj_u) {
            uint32_t *st = p.rng + (size_t)row * 16, rs[6], o[4];
#pragma unroll
            for (int i = 0; i < 6; ++i) rs[i] = st[i];
            philox4x32_10(rs[2], rs[3], rs[4], rs[5], rs[0], rs[1], o);
            if (lane == 0) {
                s.rand64 = ((uint64_t)o[0] << 32) | o[1];
                st[2] = rs[2] + 1u;
                if (rs[2] + 1u == 0u) st[3] = rs[3] + 1u;
            }
        }
        __syncthreads();
        return;
    }

    // the slices' masses in the row's frame: lane l holds slice l, or slices 2l and 2l + 1 of a row of more than 64
    constexpr int kAhead = 4;                            // sums asked for before the frames are known: slices up to 3 octaves below the row's
    const PartHdr *hdrs = v.hdr + (size_t)row * G;
    const uint64_t *sums = v.stash + (size_t)row * G * kStashCap;
    const uint32_t per = G > (uint32_t)kWave ? 2u : 1u;
    uint32_t key[2];
    uint4 ahead[2][kAhead];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const uint32_t g = min((uint32_t)lane * per + (uint32_t)k, G - 1u);
        key[k] = hdrs[g].mkey;
        const uint4 *q = reinterpret_cast<const uint4 *>(sums + (size_t)g * kStashCap);
#pragma unroll
        for (int d = 0; d < kAhead; ++d) ahead[k][d] = q[d];
    }
    const float xmax = fkey_inv(wave_max_u32(max(key[0], key[1])));
    const float M = __builtin_floorf(xmax);
    M96 mass[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const uint32_t g = (uint32_t)lane * per + (uint32_t)k;
        const float df = M - __builtin_floorf(fkey_inv(key[k]));
        const uint32_t d = df >= 64.0f ? 64u : (uint32_t)df;
        uint4 q = ahead[k][0];
#pragma unroll
        for (int i = 1; i < kAhead; ++i)
            if (d == (uint32_t)i) q = ahead[k][i];
        if (d >= (uint32_t)kAhead && d <= 40u) q = reinterpret_cast<const uint4 *>(sums + (size_t)min(g, G - 1u) * kStashCap)[d];
        const uint64_t lo = ((uint64_t)q.y << 32) | q.x, hi = q.z;
        mass[k] = M96{d == 0u ? lo : (lo >> (d & 63u)) | (hi << ((64u - d) & 63u)), (uint32_t)(hi >> (d & 63u))};
        if (d > 40u || (uint32_t)k >= per || g >= G) mass[k] = M96{0ull, 0u};        // 41 octaves and more below: nothing of the slice is live
    }
    const Limbs both = limbs(mass[0] + mass[1]), upto = wave_inclusive_scan(both);
    const M96 D = m96(lane_of(upto, 63u));
    __syncthreads();
    const uint64_t rand64 = uniform(s.rand64);
    const M96 r = p.inj_u ? m96(ceil_mul(p.inj_u[row], wide(D))) : m96(r_from_bits(rand64, wide(D)));
    uint32_t g;
    M96 r_in;
    {
        const M96 inc = m96(upto), exc = m96(upto - both);
        const uint32_t l = (uint32_t)__builtin_ctzll(__builtin_amdgcn_ballot_w64(inc >= r));         // 1 <= r <= D: there is one
        r_in = r - lane_of(exc, l);
        g = l * per;
        const M96 first = lane_of(mass[0], l);
        if (!(first >= r_in)) { r_in = r_in - first; g += 1u; }
    }
    if (__builtin_expect(p.e_bits != nullptr, 0)) {
        // diagnostics: the slices' e into the row's frame, dead tokens as 0
        uint4 *eb4 = reinterpret_cast<uint4 *>(p.e_bits + (int64_t)row * p.V);
        auto fix = [&](uint32_t b, uint32_t d) { b = rebase_bits(min(b, 0x3FFFFFFFu), d); return b < kEMinBits ? 0u : b; };
        for (uint32_t i4 = (uint32_t)tid; i4 < V4; i4 += kKeepT) {
            const float df = M - __builtin_floorf(fkey_inv(hdrs[i4 >> (LOG2 - 2)].mkey));
            const uint32_t d = df >= 64.0f ? 64u : (uint32_t)df;
            uint4 q = eb4[i4];
            q.x = fix(q.x, d); q.y = fix(q.y, d); q.z = fix(q.z, d); q.w = fix(q.w, d);
            eb4[i4] = q;
        }
    }
    if (__builtin_expect(p.diag != nullptr, 0)) keep_diag(p, s, row, xmax, D, rand64);

    // that slice's tokens, through LDS
    const uint32_t g0 = g << (LOG2 - 2);
    const char *lrow = logits_row(p, row);
    {
        float4 l[U];
#pragma unroll
        for (int j = 0; j < U; ++j) l[j] = load_logits4(lrow, min(g0 + (uint32_t)(j * kKeepT + tid), V4 - 1u), p.dtype);
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const uint32_t at = (uint32_t)(j * kKeepT + tid);
            s.x[at + at / (uint32_t)U] = make_float4(sf(l[j].x * p.c), sf(l[j].y * p.c), sf(l[j].z * p.c), sf(l[j].w * p.c));
        }
    }
    __syncthreads();
    auto weight = [&](float x) -> uint64_t {
        const uint32_t b = e_bits_of(x, M);
        return b >= kEMinBits ? w_of_bits(b) : 0ull;
    };
    uint64_t lo = 0, hi = 0;                             // halves summed apart: T * 2^32 at most
#pragma unroll
    for (int j = 0; j < U; ++j)
        if (g0 + (uint32_t)(tid * U + j) < V4) {         // past the end of the row: no weight
            const float4 x = s.x[tid * U + j + tid];
            const uint64_t w0 = weight(x.x), w1 = weight(x.y), w2 = weight(x.z), w3 = weight(x.w);
            lo += (w0 & 0xFFFFFFFFull) + (w1 & 0xFFFFFFFFull) + (w2 & 0xFFFFFFFFull) + (w3 & 0xFFFFFFFFull);
            hi += (w0 >> 32) + (w1 >> 32) + (w2 >> 32) + (w3 >> 32);
        }
    const Limbs mine = limbs(m96((u128)lo + ((u128)hi << 32))), run = wave_inclusive_scan(mine);
    M96 inc = m96(run);
    if (lane == kWave - 1) s.waves[wave] = inc;
    __syncthreads();
    if (wave) {
        const Limbs before = wave_inclusive_scan(limbs(lane < wave ? s.waves[lane] : M96{0ull, 0u}));
        inc = inc + m96(lane_of(before, 63u));
    }
    const M96 exc = inc - m96(mine);
    const uint64_t vote = __builtin_amdgcn_ballot_w64(exc < r_in && inc >= r_in);
    if (vote == 0ull) return;                            // another wave's thread owns the target
    const uint32_t o = (uint32_t)__builtin_ctzll(vote), t0 = (uint32_t)(wave * kWave) + o;
    const M96 r2 = r_in - lane_of(exc, o);
    const uint32_t at = t0 * (uint32_t)U + ((uint32_t)lane >> 2);
    uint64_t w = 0;
    if (lane < T && g0 + at < V4) {
        const float4 q = s.x[at + t0];
        const uint32_t c = (uint32_t)lane & 3u;
        w = weight(c == 0u ? q.x : c == 1u ? q.y : c == 2u ? q.z : q.w);
    }
    const Limbs one = limbs(M96{w, 0u}), sofar = wave_inclusive_scan(one);
    if (m96(sofar - one) < r2 && m96(sofar) >= r2) {
        const int32_t pick = (int32_t)((g0 + at) * 4u + ((uint32_t)lane & 3u));
        p.out[row] = pick;
        if (p.diag) p.diag[row].index = pick;
    }
}

// The streaming pass for calls with penalties too large for the one-launch path: logits and penalties
// are read once, x = sf((sf(l) - pen) * c) as in the cluster kernel, everything after that is the
// streaming pass.  The sampled token is not known yet, but every OTHER token's new penalty is
// fma(pen, decay, 0), so the pass writes those from its registers -- 12 bytes per token in all, as the
// reference's single kernel moves (sampling.cu:211,220,427-437) -- and the finishing workgroup patches the
// one sampled token.  That needs the sampled token's old value, and a row the finishing workgroup has to do
// the slow way needs the old values of all its tokens; penalties are non-zero only where tokens have been
// generated, so each slice notes the old values whose bit pattern is not +0.0 (up to kPenCap - 1 of them; a
// slice with more leaves its penalties untouched and says so, and penalty_fix_kernel rewrites such slices
// once the tokens are known).  Groups of four that are all +0.0 stay +0.0 under a finite decay and are
// not written at all.
template <int R>
__global__ void __launch_bounds__(kThreads, R <= 8 ? 4 : 2) stream_pen_kernel(const Params p, const StreamView v)
{
    constexpr int kRep = stream_copies<R>();
    __shared__ LdsA<kRep> s;
    __shared__ uint64_t noted[kWaves][kPenWave];
    __shared__ uint32_t nnote[kWaves];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    const uint32_t G = v.G;
    const uint32_t row = blockIdx.x / G, part = blockIdx.x - row * G;
    const bool reporter = blockIdx.x == 0 && threadIdx.x == 0;
    PrevCall prev;
    prev.slow_rows = 0; prev.meta = 0;
    if (reporter) prev = report_begin(p);
    Slice<R, true> sl;
    slice_setup(p, sl, row, part, G);
    const float lmax = slice_load(p, sl);
    if (reporter) report_end(p, prev, true);
    if (p.defer_pen == 2) {
        // the penalties whose bit pattern is not +0.0, side by side into this wave's notes
        uint32_t fill = 0;                               // wave-uniform: every lane takes part in every vote
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const uint32_t b4[4] = {__float_as_uint(sl.pen[j].x), __float_as_uint(sl.pen[j].y), __float_as_uint(sl.pen[j].z), __float_as_uint(sl.pen[j].w)};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const bool nz = j < sl.nv && b4[q] != 0u;
                const uint64_t vote = __ballot(nz);
                if (nz) {
                    const uint32_t pos = fill + __builtin_amdgcn_mbcnt_hi((uint32_t)(vote >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)vote, 0u));
                    if (pos < (uint32_t)kPenWave) noted[wave][pos] = ((uint64_t)b4[q] << 32) | ((sl.base4 + (uint32_t)j * kThreads) * 4u + (uint32_t)q);
                }
                fill += (uint32_t)__popcll(vote);
            }
        }
        if (lane == 0) nnote[wave] = fill;
        __syncthreads();
        uint32_t total = 0, before = 0;
        bool fits = true;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const uint32_t n = nnote[w];
            if (w < wave) before += n;
            total += n;
            fits = fits && n <= (uint32_t)kPenWave;
        }
        fits = fits && total < (uint32_t)kPenCap;
        uint64_t *rec = v.pens + ((size_t)row * G + part) * v.pen_stride;
        if (fits) {
            for (uint32_t i = (uint32_t)lane; i < fill; i += kWave) rec[1 + before + i] = noted[wave][i];
            if (tid == 0) rec[0] = total;
#pragma unroll
            for (int j = 0; j < R; ++j) {
                float4 q = sl.pen[j];
                if (j < sl.nv && (__float_as_uint(q.x) | __float_as_uint(q.y) | __float_as_uint(q.z) | __float_as_uint(q.w)) != 0u) {
                    q.x = __builtin_fmaf(q.x, p.decay, 0.0f); q.y = __builtin_fmaf(q.y, p.decay, 0.0f);
                    q.z = __builtin_fmaf(q.z, p.decay, 0.0f); q.w = __builtin_fmaf(q.w, p.decay, 0.0f);
                    sl.pn4[sl.base4 + (uint32_t)j * kThreads] = q;
                }
            }
        } else if (tid == 0) rec[0] = kPenDeferred;
    }
    slice_count_and_stash<R, kThreads, kRep, false, false, R == 8 ? kPenStashCap : kStashCap>(p, v, s, sl.eb, lmax, row, part, sl.base4, sl.nv);
}

// pen <- fma(pen, decay, onehot * (pen == 0 ? presence : repetition)), the switch on the value before
// the decay (reference: sampling.cu:427-437), from the sampled token in p.out, for the slices that still
// hold their old penalties: all of them when the streaming pass left the penalties alone (defer_pen 1),
// else those marked deferred -- by the pass (too many non-zero penalties to note) or by the finishing
// workgroup of a row done the slow way (which played the notes back).  One workgroup per slice; the others
// leave after one load.
template <int R>
__global__ void __launch_bounds__(kThreads) penalty_fix_kernel(const Params p, const StreamView v)
{
    const uint32_t G = v.G;
    const uint32_t row = blockIdx.x / G, part = blockIdx.x - row * G;
    if (p.defer_pen == 2 && !(v.pens[((size_t)row * G + part) * v.pen_stride] & kPenDeferred)) return;
    const uint32_t V4 = (uint32_t)p.V >> 2;
    const uint32_t idx = (uint32_t)p.out[row];
    float4 *pn4 = reinterpret_cast<float4 *>(p.penalties + (int64_t)row * p.V);
    const uint32_t base4 = part * (uint32_t)(kThreads * R) + threadIdx.x;
    float4 q[R];
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const uint32_t i4 = base4 + (uint32_t)j * kThreads;
        if (i4 < V4) q[j] = pn4[i4];
    }
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const uint32_t i4 = base4 + (uint32_t)j * kThreads;
        if (i4 < V4) {
            float4 w = q[j];
            const uint32_t e0 = i4 * 4;
            w.x = __builtin_fmaf(w.x, p.decay, (e0 + 0 != idx) ? 0.0f : (w.x == 0.0f ? p.presence : p.repetition));
            w.y = __builtin_fmaf(w.y, p.decay, (e0 + 1 != idx) ? 0.0f : (w.y == 0.0f ? p.presence : p.repetition));
            w.z = __builtin_fmaf(w.z, p.decay, (e0 + 2 != idx) ? 0.0f : (w.z == 0.0f ? p.presence : p.repetition));
            w.w = __builtin_fmaf(w.w, p.decay, (e0 + 3 != idx) ? 0.0f : (w.w == 0.0f ? p.presence : p.repetition));
            pn4[i4] = w;
        }
    }
}

// ------------------------------------------------------------ one-launch path --
// The streaming pass and the finish in ONE launch, for calls small enough that a second and a third
// launch (and the cold start of the finishing workgroup) cost as much as the work itself, and for
// calls with penalties, whose every workgroup holds its penalties in registers and rewrites them from there.  A row is worked by G workgroups (logical ids follow the order in which workgroups
// start once the launch is larger than the GPU holds at once).  Each reads its slice once, publishes
// the slice's record exactly as the streaming pass does -- with device-scope atomic stores -- and
// counts itself in (release).  The workgroup that arrives last finishes the row from the records
// (acquire; finish_row) and posts a verdict: the sampled token, or "fall back".  The others wait for
// the verdict -- that is the only wait, and it is for a workgroup that is already running.  On "fall
// back" (a nucleus or a tie too large for the stashes) all G workgroups go on with the cluster path's
// rounds from the tokens they still hold in registers: the row's level-1 histogram is already
// complete in memory, so they start at the boundary search.  With penalties the workgroups that wait write
// theirs, decayed, while they do, the last one once it has posted the verdict; the sampled token's is written again when
// it is known.  The last workgroup to leave cleans the row's record.
template <int R, bool PEN>
struct FusedLds {
    union {
        LdsA<stream_copies<R>()> a;
        struct { Lds s; LdsB t; } f;
    };
};

template <int R, bool PEN>
__device__ __forceinline__ bool fused_fallback(const Params &p, const StreamView &v, Lds &s, Slice<R, PEN> &sl, uint32_t slice_key)
{
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    const uint32_t G = sl.G, row = sl.row, part = sl.part;
    RowCtl *rc = sl.rc;
    draw_rand(p, s, row);
    // the slices' maxima, the row's level-1 histogram (complete: every workgroup has arrived) and
    // this slice's own bins, all as they were published
    uint32_t mk = 0;
    if ((uint32_t)tid < G) mk = (uint32_t)a_load(reinterpret_cast<const uint64_t *>(&v.hdr[(size_t)row * G + tid]));
    const uint64_t g0 = a_load(&rc->h[0][tid]), g1 = a_load(&rc->h[0][tid + kThreads]);
    uint64_t mine = 0;
    if (tid < kSB) mine = a_load(&v.shist[((size_t)row * G + part) * kSB + tid]);
    uint32_t kmax, kmin;
    {
        const uint32_t a = wave_max_u32(mk), b = wave_max_u32((uint32_t)tid < G ? ~mk : 0u);
        __syncthreads();
        if (lane == 0) { s.u32[wave] = a; s.u32[kWaves + wave] = b; }
        __syncthreads();
        kmax = s.u32[0]; kmin = s.u32[kWaves];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) { kmax = max(kmax, s.u32[w]); kmin = max(kmin, s.u32[kWaves + w]); }
        kmin = ~kmin;
    }
    const float M = __builtin_floorf(fkey_inv(kmax)), Mloc = __builtin_floorf(fkey_inv(slice_key));
    const float dd = M - Mloc;
    const uint32_t delta = dd >= 64.0f ? 64u : (uint32_t)dd;
    // the registers hold e unclamped in the slice's frame: into the row's frame, dead tokens at 2^-41
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
        for (int k = 0; k < 4; ++k) sl.eb[j * 4 + k] = rebase_bits(min(sl.eb[j * 4 + k], 0x3FFFFFFFu), delta);
    sl.kmax_row = kmax;
    sl.h_used = 1u;                                      // the row's level-1 histogram is to be cleared
    sl.mx_posted = false;
    auto clear_used = [&]() {
        for (uint32_t i = 0; i <= (uint32_t)kLevels; ++i)
            if (sl.h_used >> i & 1u) zero_slice(rc->h[i], (i == 0u || i == (uint32_t)kLevels) ? (uint32_t)kNB : 128u, part, G);
        sl.h_used = 0u;
    };
    if (M - __builtin_floorf(fkey_inv(kmin)) < 88.0f) {
        // positions by absolute octave are unambiguous: both histograms into the row's frame
        const uint32_t m4 = (uint32_t)(int)(M - 128.0f * __builtin_floorf(M * 0.0078125f)) * 4u;
        const uint32_t r0 = ((uint32_t)tid + 160u - m4) & 511u, r1 = ((uint32_t)tid + kThreads + 160u - m4) & 511u;
        for (int b = tid; b < kNB; b += kThreads) { s.g[b] = 0; s.hm[b] = 0; }
        __syncthreads();
        if (r0 < 164u) s.g[kBin0 + r0] = g0;
        if (r1 < 164u) s.g[kBin0 + r1] = g1;
        if (tid < kSB && (uint32_t)tid >= 4u * delta && delta < 64u) s.hm[kBin0 + (uint32_t)tid - 4u * delta] = mine;
        __syncthreads();
    } else {
        // slices too far apart for shared positions: level 1 again, in the row's frame, through the
        // spare histogram (every token is counted, dead ones too, so that the counts add up)
        __syncthreads();
        lds_hist_zero(s, kNB);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < R; ++j)
            if (j < sl.nv) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t b = opaque(sl.eb[j * 4 + k]);
                    lds_hist_add(s, b >> 21, b);
                }
            }
        if (!hist_combine(s, p.hdr, G, rc->h[kLevels], kNB, (uint32_t)p.V, lane, wave)) return false;
        clear_used();                                    // every workgroup has read the first histogram before it published this one
        sl.h_used = 1u << kLevels;
    }
    return slice_finish(p, s, sl);
}

// PRE: slices per wave whose first tokens the finishing workgroup asks for ahead (the host's choice, as for finish_kernel).
// With 16 whatever the row and the random number drawn before the slice was asked for, 320 rows of 8192 tokens, two slices
// each, N(0,2) with 16 large logits in 4096, top_k 50, took 19.0 us a call; 17.4 this way.
template <int R, bool PEN, int PRE>
__global__ void __launch_bounds__(kThreads, 2) fused_kernel(const Params p, const StreamView v)
{
    constexpr int kRep = stream_copies<R>();
    static_assert(R == 4 || R == 8 || R == 16, "slices of 4096, 8192 or 16384 tokens");
    __shared__ FusedLds<R, PEN> u;
    const int tid = threadIdx.x;
    const uint32_t G = v.G;
    // logical id: the hardware's while the device holds the whole launch at once (every call routed here
    // by itself does), else a ticket, so that a row's workgroups are always the next ones to start
    uint32_t id = blockIdx.x;
    constexpr uint32_t kResident = 256u * (R == 16 && PEN ? 2u : 3u);     // workgroups of this kernel the device holds at once
    if (gridDim.x > kResident) {
        if (tid == 0) {
            u.a.u32[8] = take_ticket(p.hdr);
        }
        __syncthreads();
        id = u.a.u32[8];
    }
    const uint32_t row = id / G, part = id - row * G;
    Slice<R, PEN> sl;
    slice_setup(p, sl, row, part, G);
    RowCtl *rc = sl.rc;
    // the row's generator state is asked for ahead of the slice and used behind it
    uint32_t rs[6] = {0u, 0u, 0u, 0u, 0u, 0u};
    uint32_t *st = p.rng + (size_t)row * 16;
    if (tid == kWave && !p.inj_u) {
#pragma unroll
        for (int i = 0; i < 6; ++i) rs[i] = st[i];
    }
    // the call's first thread reports on the streaming call before it, if there was one (report_begin)
    const bool reporter = blockIdx.x == 0 && tid == 0 && p.host_words != nullptr;
    PrevCall prev;
    prev.slow_rows = 0; prev.meta = 0;
    if (reporter) prev = report_begin(p);
    const float lmax = slice_load(p, sl);
    if (reporter) report_end(p, prev, false);
    const uint32_t key = slice_count_and_stash<R, kThreads, kRep, true>(p, v, u.a, sl.eb, lmax, row, part, sl.base4, sl.nv);

    // Count this slice in.  Everything it published went out as device-scope atomic stores (written
    // through to the level all XCDs share) and has been acknowledged before the count is raised; the
    // finishing workgroup reads with device-scope atomic loads.  No cache write-back or invalidation
    // is needed for that, and none is asked for: a release here would write back the whole L2.
#ifndef RS_FUSED_RELAXED
#define RS_FUSED_RELAXED 1
#endif
    // the row's random number, should this workgroup be the one that finishes the row: drawn while the stores are on their way
    uint64_t drawn = 0;
    if (tid == kWave && !p.inj_u) {
        uint32_t o[4];
        philox4x32_10(rs[2], rs[3], rs[4], rs[5], rs[0], rs[1], o);
        drawn = ((uint64_t)o[0] << 32) | o[1];
    }
    wait_vmem();
    __syncthreads();
    if (tid == 0)
        u.a.u32[9] = RS_FUSED_RELAXED ? __hip_atomic_fetch_add(&rc->arrived, 1u, __ATOMIC_RELAXED, RS_AGENT)
                                      : __hip_atomic_fetch_add(&rc->arrived, 1u, __ATOMIC_ACQ_REL, RS_AGENT);
    __syncthreads();
    const bool last = u.a.u32[9] == G - 1u;
    __syncthreads();                                     // the LDS of the streaming pass is given up here
    Lds &s = u.f.s;
    LdsB &t = u.f.t;
    if (tid == 0) { s.abort = 0; s.host_words = p.host_words; s.who = row << 16 | part; s.seen = 0; s.want = 0; }
    // Every penalty but the sampled token's becomes fma(pen, decay, 0) whatever is sampled: the workgroups that wait write theirs
    // while they do, the last one behind its verdict.  Groups of four that are all +0.0 stay that under a finite decay.  (Written
    // behind the verdict, all of them: 32 rows of 131072 20.8 us a call, 19.4 this way.)  A row that falls back writes them once more.
    // A workgroup whose wait gives up puts its penalties back: no token was sampled for it.
    auto rewrite = [&](auto fn) {
        if constexpr (PEN) {
            const bool finite = p.decay - p.decay == 0.0f;
#pragma unroll
            for (int j = 0; j < R; ++j) {
                const float4 q = sl.pen[j];
                if (j < sl.nv && (!finite || (__float_as_uint(q.x) | __float_as_uint(q.y) | __float_as_uint(q.z) | __float_as_uint(q.w)) != 0u))
                    sl.pn4[sl.base4 + (uint32_t)j * kThreads] = make_float4(fn(q.x), fn(q.y), fn(q.z), fn(q.w));
            }
        }
    };
    auto decayed = [&]() { rewrite([&](float q) { return __builtin_fmaf(q, p.decay, 0.0f); }); };
    auto put_back = [&]() { rewrite([](float q) { return q; }); };
    uint32_t verdict = 0;
    bool gave_up = false;
    if (last) {
        // the token list: the cluster rounds' histogram copies, which are not in use while a row is
        // finished from the stashes (no dynamic LDS in this kernel: see rs_sample_ex)
        static_assert(sizeof(s.hr) == 2048 * sizeof(uint64_t), "room for a list of 2048 tokens");
        const bool done = finish_row<kThreads, PRE, true>(p, v, s, t, s.hr, row, drawn);
        if (done && tid == kWave && !p.inj_u) {
            st[2] = rs[2] + 1u;                          // the row is finished: this draw is used up
            if (rs[2] + 1u == 0u) st[3] = rs[3] + 1u;
        }
        __syncthreads();
        verdict = done && t.result != 0u ? t.result : kVerdictFallback;
        if (tid == 0) a_store(&rc->verdict, verdict);
        decayed();
    } else {
        decayed();
        __syncthreads();
        if (tid == 0) {
            const uint64_t t0 = wall_clock64();
            uint32_t spins = 0, w;
            while ((w = a_load(&rc->verdict)) == 0u) {
                __builtin_amdgcn_s_sleep(2);
                if ((++spins & 255u) == 0 && (uint64_t)wall_clock64() - t0 > spin_limit(p.hdr)) { give_up(s, p.hdr, 6u); break; }
            }
            s.bc32[7] = w;
        }
        __syncthreads();
        gave_up = s.abort != 0u;
        verdict = gave_up ? kVerdictFallback : s.bc32[7];
    }
    if (verdict == kVerdictFallback) {
        // (ends with the cluster path's own leaving protocol; a wait that gives up there comes before its write of the penalties)
        if (gave_up || !fused_fallback<R, PEN>(p, v, s, sl, key)) put_back();
        return;
    }
    const uint32_t idx = verdict - 1u;
    if (PEN) {
        // the sampled token's penalty, by the thread that wrote its group before (reference: sampling.cu:427-437)
#pragma unroll
        for (int j = 0; j < R; ++j)
            if (sl.base4 + (uint32_t)j * kThreads == idx >> 2 && j < sl.nv) {
                const uint32_t q = idx & 3u;
                const float old = q == 0u ? sl.pen[j].x : q == 1u ? sl.pen[j].y : q == 2u ? sl.pen[j].z : sl.pen[j].w;
                reinterpret_cast<float *>(sl.pn4)[idx] = __builtin_fmaf(old, p.decay, old == 0.0f ? p.presence : p.repetition);
            }
    }
    // leave: the last workgroup out of the row puts its record back to zero
    __syncthreads();
    if (tid == 0) s.bc32[0] = __hip_atomic_fetch_add(&rc->done, 1u, __ATOMIC_RELAXED, RS_AGENT);
    __syncthreads();
    if (s.bc32[0] == G - 1u) {
        a_store(&rc->h[0][tid], (uint64_t)0); a_store(&rc->h[0][tid + kThreads], (uint64_t)0);
        if (tid == 0) { a_store(&rc->done, 0u); a_store(&rc->arrived, 0u); a_store(&rc->verdict, 0u); }
    }
}

}  // namespace rs
