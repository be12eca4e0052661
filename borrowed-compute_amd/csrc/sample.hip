// The next-token pick on the device: bc-infer's sampler (crates/bc-infer/src/sample.rs:24-71),
// the step after the logits head (gpu/mod.rs:499-508), with the reference's results index for
// index.
//
// Temperature 0: the first index of the highest score (sample.rs:24-32), a parallel argmax
// whose ties go to the lower index. Otherwise, per row (sample.rs:35-71):
//   max = the largest non-NaN score; p_i = exp((s_i - max) / T) with exp correctly rounded
//     (computed in double, as the CPU restatement does; the reference leaves exp to libm);
//   total = sum of p_i in index order, from -0;
//   the stable descending sort by f32::total_cmp: ascending 64-bit keys, the p key of the total
//     order inverted over the index;
//   keep = the shortest sorted prefix whose running mass (sum of p / total, each step
//     rounded) reaches top_p, at least 1; r = uniform(seed ^ step * golden) * (sum of the kept
//     p, in order); the first kept token whose running r -= p reaches <= 0, else the first.
//
// The sums are defined by their serial order, each step rounded to nearest even, but need no
// serial loop (run_chunk): while a running sum of non-negative terms stays within one binade,
// a step adds an integer of that binade's ulps, the term in ulps rounded, and only a term
// whose fraction is exactly one half depends on what came before, by the parity it meets. So
// a term is a pair of integers (for an even and an odd sum before it), pairs compose
// associatively, and a scan over the workgroup gives every partial sum exactly. The thread at
// which the sum would leave the binade (or reach the target looked for) adds its few terms one
// by one, and the scan goes on behind it with the new binade's ulp. (One lane adding 151936
// terms took 1.2 ms.)
//
// Only the kept prefix has to be sorted: a histogram of p by its leading bits bounds it from
// below (smp_margin), the tokens above the bound are compacted in index order and sorted in LDS
// (a stable radix sort through memory if they are many). Where the margin leaves no bound (top_p
// near 1) the whole row is sorted by rocPRIM.
#include <cstring>  // before rocPRIM, whose iterator header calls memset

#include <rocprim/device/device_radix_sort.hpp>

#include "common.hpp"
#include "internal.hpp"

#include <math.h>

namespace bchip {

constexpr int SMP_THREADS = 1024;

// f32::total_cmp as an unsigned key: ascending keys are ascending total order.
__device__ __forceinline__ uint32_t total_key(float x) {
    const uint32_t b = __float_as_uint(x);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float from_total_key(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// Sort key of token i: descending total order of its p, then ascending index (the stable sort).
__device__ __forceinline__ uint64_t sort_key(float p, uint32_t i) {
    return ((uint64_t)(~total_key(p)) << 32) | i;
}
__device__ __forceinline__ float key_weight(uint64_t k) { return from_total_key(~(uint32_t)(k >> 32)); }

// sample.rs:74-81.
__device__ __forceinline__ float uniform(uint64_t seed) {
    uint64_t z = seed + 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    z ^= z >> 31;
    return (float)(z >> 40) / (float)(1ull << 24);
}

// The highest score of a row and its first index: the reference's argmax starts from index 0
// and moves only on a strictly higher score, so a NaN never wins past index 0, and a row whose
// first score is NaN answers 0.
__global__ __launch_bounds__(SMP_THREADS) void k_argmax(const float* __restrict__ scores, uint32_t vocab,
                                                        uint32_t* __restrict__ ids) {
    __shared__ float bv_s[SMP_THREADS / 64];
    __shared__ uint32_t bi_s[SMP_THREADS / 64];
    const float* s = scores + (size_t)blockIdx.x * vocab;
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    float bv = -INFINITY;
    uint32_t bi = 0xffffffffu;
    for (uint32_t i = tid; i < vocab; i += SMP_THREADS) {
        const float v = s[i];
        if (v > bv) {  // strict: the first occurrence in this thread's ascending indices
            bv = v;
            bi = i;
        }
    }
    auto better = [](float v, uint32_t i, float bv, uint32_t bi) { return v > bv || (v == bv && i < bi); };
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
        const float ov = __shfl_xor(bv, d);
        const uint32_t oi = __shfl_xor(bi, d);
        if (better(ov, oi, bv, bi)) {
            bv = ov;
            bi = oi;
        }
    }
    if (lane == 0) {
        bv_s[w] = bv;
        bi_s[w] = bi;
    }
    __syncthreads();
    if (tid == 0) {
        for (int j = 1; j < SMP_THREADS / 64; j++)
            if (better(bv_s[j], bi_s[j], bv, bi)) {
                bv = bv_s[j];
                bi = bi_s[j];
            }
        // No score above -inf (or only NaN past index 0), or a NaN at index 0: index 0.
        ids[blockIdx.x] = (bi == 0xffffffffu || isnan(s[0])) ? 0u : bi;
    }
}

// Rows of at least this many tokens get the histogram that bounds the kept prefix (it sits in the
// row's key space until the keys are written).
constexpr uint32_t SMP_BINS = 4096;
constexpr uint32_t SMP_HIST_MIN = 4096;
constexpr uint32_t SMP_LDS_KEYS = 8192;  // keys sorted in LDS
constexpr uint32_t SMP_BLOCK = 4096;     // tokens a workgroup of the parallel passes
constexpr int SMP_EPT = 8;               // terms a thread of a chunk: 8192 a chunk

__device__ __forceinline__ uint32_t p_bin(float p) { return min(__float_as_uint(p) >> 18, SMP_BINS - 1u); }  // p in [0, 1]

// How far past top_p the histogram's mass of the candidates must reach, so that the f32 running
// mass over them reaches top_p for certain: four f32 sums of at most vocab non-negative terms
// are between the two (the bins, all bins, total, the mass itself), each within vocab 2^-24 of
// its size, and 1/256 covers the rest (the shares' rounding, the sums' second order).
__host__ __device__ inline float smp_margin(uint32_t vocab) { return 4.0f * 5.9604645e-8f * (float)vocab + 0.00390625f; }

// Max of each block of a row; clears the row's histogram and NaN flag.
__global__ __launch_bounds__(256) void k_sample_max(const float* __restrict__ scores, uint32_t vocab,
                                                    float* __restrict__ maxes, uint32_t* __restrict__ flags,
                                                    uint64_t* __restrict__ keys, bool hist) {
    __shared__ float red[4];
    const uint32_t tid = threadIdx.x, row = blockIdx.y, nb = gridDim.x;
    const float* s = scores + (size_t)row * vocab;
    const uint32_t c0 = blockIdx.x * SMP_BLOCK, c1 = min(c0 + SMP_BLOCK, vocab);
    float mx = -INFINITY;
    for (uint32_t i = c0 + tid; i < c1; i += 256) mx = fmaxf(mx, s[i]);  // f32::max skips NaN
#pragma unroll
    for (int d = 1; d < 64; d *= 2) mx = fmaxf(mx, __shfl_xor(mx, d));
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    if (tid == 0) {
        maxes[(size_t)row * nb + blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        if (blockIdx.x == 0) flags[row] = 0u;
    }
    if (hist) {
        float* h = (float*)(keys + (size_t)row * vocab);
        for (uint32_t i = blockIdx.x * 256 + tid; i < SMP_BINS; i += nb * 256) h[i] = 0.0f;
    }
}

// p of every token into p_out (rows vocab u64 apart) or, for a full sort, the sort keys; the
// histogram of mass by leading bits (its sums' rounding only moves the bound).
__global__ __launch_bounds__(256) void k_sample_p(const float* __restrict__ scores, uint32_t vocab, float temperature,
                                                  const float* __restrict__ maxes, uint32_t* __restrict__ flags,
                                                  uint64_t* __restrict__ keys, uint64_t* __restrict__ p_out, bool hist,
                                                  bool full) {
    __shared__ float h[SMP_BINS];
    const uint32_t tid = threadIdx.x, row = blockIdx.y, nb = gridDim.x;
    const float* s = scores + (size_t)row * vocab;
    uint64_t* kr = keys + (size_t)row * vocab;
    float* pr = (float*)(p_out + (size_t)row * vocab);
    float mx = -INFINITY;
    for (uint32_t i = tid & 63; i < nb; i += 64) mx = fmaxf(mx, maxes[(size_t)row * nb + i]);
#pragma unroll
    for (int d = 1; d < 64; d *= 2) mx = fmaxf(mx, __shfl_xor(mx, d));
    if (hist)
        for (uint32_t i = tid; i < SMP_BINS; i += 256) h[i] = 0.0f;
    __syncthreads();
    const uint32_t c0 = blockIdx.x * SMP_BLOCK, c1 = min(c0 + SMP_BLOCK, vocab);
    bool nan = false;
    for (uint32_t i = c0 + tid; i < c1; i += 256) {
        const float p = (float)exp((double)((s[i] - mx) / temperature));
        nan = nan || isnan(p);
        if (full) kr[i] = sort_key(p, i);
        else pr[i] = p;
        if (hist && p > 0.0f) atomicAdd(&h[p_bin(p)], p);
    }
    if (nan) flags[row] = 1u;
    if (hist) {
        __syncthreads();
        float* g = (float*)kr;
        for (uint32_t i = tid; i < SMP_BINS; i += 256)
            if (h[i] != 0.0f) atomicAdd(&g[i], h[i]);
    }
}

// A serial f32 sum's state and the workgroup's scratch for a scan.
struct SmpScan {
    uint2 wave[SMP_THREADS / 64];
    float sum;
    uint32_t next, found;
    uint32_t first[2];  // the first thread out of the binade, by turns
};

// Terms in ulps (for an even and for an odd running sum), composed left to right. Saturated:
// 2^26 ulps always leave the binade.
__device__ __forceinline__ uint2 compose(uint2 a, uint2 b) {
    const uint32_t lim = 1u << 26;
    const uint32_t x = a.x + ((a.x & 1u) ? b.y : b.x), y = a.y + ((a.y & 1u) ? b.x : b.y);
    return uint2{min(x, lim), min(y, lim)};
}

// Adds (SUB: subtracts) a chunk of terms, thread t's v[0 .. SMP_EPT) after thread t - 1's, to the
// serial sum in sc.sum, every step rounded as f32 rounds it. Stops behind the term at which the
// sum reaches target (SUB: is <= 0): returns its thread * SMP_EPT + index, else -1 (to every
// thread). Terms are >= 0 and not NaN (those past the list 0, which move no sum); at: the
// thread's terms of the list. SUB: the sum starts > 0 or stops at its first term. Bound by the
// workgroup's latencies, about 1.5 us a scan: one a chunk and one a binade left.
template <bool SUB, bool TARGET>
__device__ int run_chunk(SmpScan& sc, const float (&v)[SMP_EPT], int n, float target) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    __syncthreads();  // every thread is done with the last chunk's answer (and sc.sum is set)
    if (tid == 0) {
        sc.next = 0;
        sc.found = sc.first[0] = sc.first[1] = 0xffffffffu;
    }
    __syncthreads();
    for (uint32_t turn = 0;; turn ^= 1u) {
        const uint32_t t0 = sc.next;
        const float s0 = sc.sum;
        const uint32_t bits = __float_as_uint(s0) & 0x7fffffffu;
        const int e = (int)max(bits >> 23, 1u);
        const uint32_t m = (bits & 0x7fffffu) | (bits >> 23 ? 0x800000u : 0u);  // s0 = m ulps of 2^(e - 150)
        // The thread's terms in ulps: the mantissa shifted by the exponents' difference k, the bits
        // shifted out against one half.
        uint32_t q[SMP_EPT], ties = 0, sum = 0;
#pragma unroll
        for (int j = 0; j < SMP_EPT; j++) {
            const uint32_t vb = __float_as_uint(v[j]), ve = vb >> 23;
            const uint32_t vm = (vb & 0x7fffffu) | (ve ? 0x800000u : 0u);
            const int k = e - (int)max(ve, 1u);
            const uint32_t r = (uint32_t)min(max(k, 0), 25), half = (1u << r) >> 1, rem = vm & ((1u << r) - 1u);
            q[j] = (vm << (uint32_t)min(max(-k, 0), 1)) >> r;  // (a term of more binades leaves this one)
            q[j] += rem > half ? 1u : 0u;
            if (k > 0 && rem == half) ties |= 1u << j;
            sum += q[j];
        }
        uint2 a = uint2{sum, sum};
        if (ties) {
            a = uint2{0u, 0u};
#pragma unroll
            for (int j = 0; j < SMP_EPT; j++)
                a = compose(a, ties >> j & 1u ? uint2{q[j] + (q[j] & 1u), q[j] + 1u - (q[j] & 1u)} : uint2{q[j], q[j]});
        }
        if (tid < t0) a = uint2{0u, 0u};
#pragma unroll
        for (int d = 1; d < 64; d *= 2) {
            const uint2 o = uint2{__shfl_up(a.x, d), __shfl_up(a.y, d)};
            if (lane >= (uint32_t)d) a = compose(o, a);
        }
        if (lane == 63) sc.wave[w] = a;
        __syncthreads();
        uint2 wt = sc.wave[lane & (SMP_THREADS / 64 - 1)];  // the waves' totals, scanned by 16 lanes
#pragma unroll
        for (int d = 1; d < SMP_THREADS / 64; d *= 2) {
            const uint2 o = uint2{__shfl_up(wt.x, d), __shfl_up(wt.y, d)};
            if (lane >= (uint32_t)d) wt = compose(o, wt);
        }
        const uint2 before = uint2{__shfl(wt.x, (int)w - 1), __shfl(wt.y, (int)w - 1)};
        const uint2 upto = w ? compose(before, a) : a;
        const uint32_t c = (m & 1u) ? upto.y : upto.x;
        // Past this thread's terms the sum is m + c (m - c) ulps, if it is within the binade.
        bool out;
        uint32_t past;
        if constexpr (SUB) {
            out = m < c + (e == 1 ? 1u : 0x800001u);
            past = m - c;
        } else {
            out = m + c >= 0x1000000u;
            past = m + c;
        }
        // past ulps as f32: in the binade of s0 (or, below it, subnormal: exponent bits 0).
        const float after = __uint_as_float(past & 0x800000u ? ((uint32_t)e << 23) | (past & 0x7fffffu) : past);
        out = tid >= t0 && (out || (TARGET && !SUB && after >= target));
        const uint64_t b = __ballot(out);
        if (b && lane == 0) atomicMin(&sc.first[turn], 64 * w + (uint32_t)__builtin_ctzll(b));
        __syncthreads();
        const uint32_t f = sc.first[turn];
        // The sum before thread f (its predecessor's `after`), or the chunk's end.
        if (f == 0xffffffffu ? tid == SMP_THREADS - 1 : (f > t0 && tid == f - 1)) sc.sum = after;
        if (f == 0xffffffffu) {
            __syncthreads();
            return -1;
        }
        __syncthreads();
        if (tid == f) {
            float s = sc.sum;
            for (int j = 0; j < SMP_EPT; j++) {
                if (j >= n) break;
                s = SUB ? s - v[j] : s + v[j];
                if (TARGET && (SUB ? s <= 0.0f : s >= target)) {
                    sc.found = f * SMP_EPT + (uint32_t)j;
                    break;
                }
            }
            sc.sum = s;
            sc.next = f + 1;
            sc.first[turn] = 0xffffffffu;
        }
        __syncthreads();
        if (TARGET && sc.found != 0xffffffffu) return (int)sc.found;
        if (f == SMP_THREADS - 1) return -1;
    }
}

// Stable ascending radix sort of n keys by their upper 32 bits, by one workgroup through memory
// (a, then b, in turn; the result in a).
__device__ void radix_sort_keys_wg(uint64_t* a, uint64_t* b, uint32_t n, uint32_t* base, uint32_t (*cnt)[256]) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    for (int pass = 0; pass < 4; pass++) {
        const int sh = 32 + 8 * pass;
        const uint64_t* src = pass & 1 ? b : a;
        uint64_t* dst = pass & 1 ? a : b;
        if (tid < 256) base[tid] = 0;
        __syncthreads();
        for (uint32_t i = tid; i < n; i += SMP_THREADS) atomicAdd(&base[(src[i] >> sh) & 255u], 1u);
        __syncthreads();
        if (tid == 0) {
            uint32_t run = 0;
            for (int d = 0; d < 256; d++) {
                const uint32_t k = base[d];
                base[d] = run;
                run += k;
            }
        }
        for (uint32_t i0 = 0; i0 < n; i0 += SMP_THREADS) {
            for (uint32_t k = tid; k < SMP_THREADS / 64 * 256; k += SMP_THREADS) cnt[k / 256][k % 256] = 0;
            __syncthreads();
            const bool have = i0 + tid < n;
            const uint64_t key = have ? src[i0 + tid] : 0;
            const uint32_t d = (uint32_t)(key >> sh) & 255u;
            uint64_t peers = __ballot(have);
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const uint64_t set = __ballot((d >> k) & 1u);
                peers &= (d >> k) & 1u ? set : ~set;
            }
            const uint32_t rank = (uint32_t)__popcll(peers & ((1ull << lane) - 1ull));
            if (have && rank == 0) cnt[w][d] = (uint32_t)__popcll(peers);
            __syncthreads();
            if (have) {
                uint32_t at = base[d] + rank;
                for (uint32_t k = 0; k < w; k++) at += cnt[k][d];
                dst[at] = key;
            }
            __syncthreads();
            if (tid < 256)
                for (uint32_t k = 0; k < SMP_THREADS / 64; k++) base[tid] += cnt[k][tid];
            __syncthreads();
        }
        __threadfence();
        __syncthreads();
    }
}

// Per row: total, the kept prefix's candidates sorted, the nucleus and the draw. full: keys holds
// every p's key unsorted and sorted their order; else sorted holds p (f32) and keys the
// histogram.
__global__ __launch_bounds__(SMP_THREADS) void k_sample_pick(uint64_t* keys, uint64_t* sorted, uint32_t vocab,
                                                             const uint32_t* __restrict__ flags, float top_p, uint64_t seed,
                                                             uint64_t step0, uint32_t* __restrict__ ids, bool hist,
                                                             bool full) {
    __shared__ SmpScan sc;
    __shared__ uint64_t ks[SMP_LDS_KEYS];
    __shared__ uint32_t cnt[SMP_THREADS / 64][256], base[256], wsum[SMP_THREADS / 64];
    __shared__ float fsum[SMP_THREADS / 64];
    __shared__ uint64_t best[SMP_THREADS / 64];
    __shared__ uint32_t bound_s;
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6, row = blockIdx.x;
    uint64_t* kr = keys + (size_t)row * vocab;
    uint64_t* sr = sorted + (size_t)row * vocab;
    const float* pr = (const float*)sr;
    auto p_at = [&](uint32_t i) { return full ? key_weight(kr[i]) : pr[i]; };
    if (flags[row]) {
        // A NaN: total and every running mass are NaN, nothing is reached, and the pick is the first
        // of the order.
        uint64_t k = ~0ull;
        for (uint32_t i = tid; i < vocab; i += SMP_THREADS) k = min(k, full ? kr[i] : sort_key(pr[i], i));
#pragma unroll
        for (int d = 1; d < 64; d *= 2) k = min(k, (uint64_t)__shfl_xor((unsigned long long)k, d));
        if (lane == 0) best[w] = k;
        __syncthreads();
        if (tid == 0) {
            for (uint32_t j = 1; j < SMP_THREADS / 64; j++) k = min(k, best[j]);
            ids[row] = (uint32_t)k;
        }
        return;
    }
    // The lowest bin of the candidates: the mass of the bins from it up passes top_p by the margin.
    uint32_t bound = 0;
    if (hist) {
        constexpr uint32_t BPT = SMP_BINS / SMP_THREADS;
        const float* h = (const float*)kr;
        float bin[BPT], mine = 0.0f;  // thread t: bins from the top down
#pragma unroll
        for (uint32_t k = 0; k < BPT; k++) {
            bin[k] = h[SMP_BINS - 1u - (BPT * tid + k)];
            mine += bin[k];
        }
        float run = mine;
#pragma unroll
        for (int d = 1; d < 64; d *= 2) {
            const float o = __shfl_up(run, d);
            if (lane >= (uint32_t)d) run += o;
        }
        if (lane == 63) fsum[w] = run;
        if (tid == 0) bound_s = 0u;
        __syncthreads();
        float all = 0.0f, before = 0.0f;
        for (uint32_t k = 0; k < SMP_THREADS / 64; k++) {
            if (k < w) before += fsum[k];
            all += fsum[k];
        }
        const float want = (top_p + smp_margin(vocab)) * all;
        float x = before + run - mine;
        if (x < want && x + mine >= want) {
#pragma unroll
            for (uint32_t k = 0; k < BPT; k++) {
                x += bin[k];
                if (x >= want) {
                    atomicMax(&bound_s, SMP_BINS - 1u - (BPT * tid + k));
                    break;
                }
            }
        }
        __syncthreads();  // (the histogram is read: the candidates' keys may take its place)
        bound = bound_s;
    }
    // total, and the candidates' keys in index order.
    uint32_t ncand = 0;
    if (tid == 0) sc.sum = -0.0f;
    for (uint32_t c0 = 0; c0 < vocab; c0 += SMP_THREADS * SMP_EPT) {
        float v[SMP_EPT];
        const uint32_t i0 = c0 + tid * SMP_EPT;
        const int n = i0 < vocab ? (int)min((uint32_t)SMP_EPT, vocab - i0) : 0;
        uint32_t take = 0;
#pragma unroll
        for (int j = 0; j < SMP_EPT; j++) {
            v[j] = j < n ? p_at(i0 + j) : 0.0f;
            if (j < n && p_bin(v[j]) >= bound) take |= 1u << j;
        }
        run_chunk<false, false>(sc, v, n, 0.0f);
        if (!full) {
            uint32_t mine = (uint32_t)__popc(take), run = mine;
#pragma unroll
            for (int d = 1; d < 64; d *= 2) {
                const uint32_t o = __shfl_up(run, d);
                if (lane >= (uint32_t)d) run += o;
            }
            if (lane == 63) wsum[w] = run;
            __syncthreads();
            uint32_t before = 0, all = 0;
            for (uint32_t k = 0; k < SMP_THREADS / 64; k++) {
                if (k < w) before += wsum[k];
                all += wsum[k];
            }
            uint32_t at = ncand + before + run - mine;
#pragma unroll
            for (int j = 0; j < SMP_EPT; j++)
                if (take >> j & 1u) {
                    const uint64_t k = sort_key(v[j], i0 + j);
                    kr[at] = k;
                    if (at < SMP_LDS_KEYS) ks[at] = k;
                    at++;
                }
            ncand += all;
            __syncthreads();
        }
    }
    const float total = sc.sum;
    __syncthreads();
    // Sorted: in LDS (ks), or in memory (list).
    const uint64_t* list = full ? sr : kr;
    bool lds = false;
    if (full) {
        ncand = vocab;
    } else if (ncand <= SMP_LDS_KEYS) {
        lds = true;
        uint32_t np = 1;
        while (np < ncand) np *= 2;
        for (uint32_t i = ncand + tid; i < np; i += SMP_THREADS) ks[i] = ~0ull;
        __syncthreads();
        for (uint32_t k = 2; k <= np; k *= 2)
            for (uint32_t j = k / 2; j > 0; j /= 2) {
                for (uint32_t x = tid; x < np / 2; x += SMP_THREADS) {
                    const uint32_t i = 2 * x - (x & (j - 1)), o = i + j;
                    const uint64_t ka = ks[i], kb = ks[o];
                    if ((ka > kb) == ((i & k) == 0)) {
                        ks[i] = kb;
                        ks[o] = ka;
                    }
                }
                __syncthreads();
            }
    } else {
        // (p is read: its space takes the sort's other half; every read of it is past)
        __threadfence();
        __syncthreads();
        radix_sort_keys_wg(kr, sr, ncand, base, cnt);
    }
    auto key_at = [&](uint32_t i) { return lds ? ks[i] : list[i]; };
    // keep: the running mass reaches top_p.
    auto load = [&](uint32_t c0, uint32_t end, float (&v)[SMP_EPT], bool share) {
        const uint32_t i0 = c0 + tid * SMP_EPT;
        const int n = i0 < end ? (int)min((uint32_t)SMP_EPT, end - i0) : 0;
#pragma unroll
        for (int j = 0; j < SMP_EPT; j++) {
            const float p = j < n ? key_weight(key_at(i0 + j)) : 0.0f;
            v[j] = share && j < n ? p / total : p;
        }
        return n;
    };
    uint32_t keep = ncand;
    bool reached = false;
    if (tid == 0) sc.sum = 0.0f;
    __syncthreads();
    for (uint32_t c0 = 0; c0 < ncand && !reached; c0 += SMP_THREADS * SMP_EPT) {
        float v[SMP_EPT];
        const int n = load(c0, ncand, v, true);
        const int at = run_chunk<false, true>(sc, v, n, top_p);
        if (at >= 0) {
            keep = c0 + (uint32_t)at + 1;
            reached = true;
        }
    }
    // The kept mass, in sorted order from -0, and the draw.
    if (tid == 0) sc.sum = -0.0f;
    __syncthreads();
    for (uint32_t c0 = 0; c0 < keep; c0 += SMP_THREADS * SMP_EPT) {
        float v[SMP_EPT];
        const int n = load(c0, keep, v, false);
        run_chunk<false, false>(sc, v, n, 0.0f);
    }
    const float kept = sc.sum;
    __syncthreads();
    const uint64_t step = step0 + row;
    if (tid == 0) sc.sum = uniform(seed ^ (step * 0x9e3779b97f4a7c15ull)) * kept;
    __syncthreads();
    uint32_t id = (uint32_t)(key_at(0) & 0xffffffffu);
    for (uint32_t c0 = 0; c0 < keep; c0 += SMP_THREADS * SMP_EPT) {
        float v[SMP_EPT];
        const int n = load(c0, keep, v, false);
        const int at = run_chunk<true, true>(sc, v, n, 0.0f);
        if (at >= 0) {
            id = (uint32_t)(key_at(c0 + (uint32_t)at) & 0xffffffffu);
            break;
        }
    }
    if (tid == 0) ids[row] = id;
}

static uint32_t sample_blocks(uint32_t vocab) { return (vocab + SMP_BLOCK - 1) / SMP_BLOCK; }

// Keys twice, the blocks' maxima, the rows' flags and the sort's own scratch.
size_t sample_scratch_bytes(uint32_t rows, uint32_t vocab) {
    size_t sort_bytes = 0;
    (void)rocprim::radix_sort_keys(nullptr, sort_bytes, (const uint64_t*)nullptr, (uint64_t*)nullptr, vocab, 0, 64);
    const size_t keys = (size_t)rows * vocab * sizeof(uint64_t);
    return 2 * keys + (size_t)rows * (sample_blocks(vocab) + 1) * sizeof(float) + ((sort_bytes + 255) & ~(size_t)255) + 1024;
}

hipError_t sample_launch(const float* scores, uint32_t rows, uint32_t vocab, float temperature, float top_p,
                         uint64_t seed, uint64_t step0, uint32_t* ids, void* scratch, size_t scratch_bytes,
                         hipStream_t s) {
    if (rows == 0 || vocab == 0) return hipSuccess;
    if (!(temperature > 0.0f)) {
        hipLaunchKernelGGL(k_argmax, dim3(rows), dim3(SMP_THREADS), 0, s, scores, vocab, ids);
        return hipGetLastError();
    }
    size_t sort_bytes = 0;
    hipError_t e = rocprim::radix_sort_keys(nullptr, sort_bytes, (const uint64_t*)nullptr, (uint64_t*)nullptr, vocab,
                                            0, 64, s);
    if (e != hipSuccess) return e;
    const size_t keys = (size_t)rows * vocab * sizeof(uint64_t);
    const uint32_t nb = sample_blocks(vocab);
    char* base = (char*)(((uintptr_t)scratch + 255) & ~(uintptr_t)255);
    uint64_t* kin = (uint64_t*)base;
    uint64_t* kout = (uint64_t*)(base + keys);
    float* maxes = (float*)(base + 2 * keys);
    uint32_t* flags = (uint32_t*)(maxes + (size_t)rows * nb);
    void* tmp = (void*)(((uintptr_t)(flags + rows) + 255) & ~(uintptr_t)255);
    if ((char*)tmp + sort_bytes > (char*)scratch + scratch_bytes) return hipErrorInvalidValue;
    // No bound within the margin: the whole row may be kept (one that fits LDS is sorted there).
    const bool bounded = top_p + smp_margin(vocab) < 1.0f;
    const bool full = !bounded && vocab > SMP_LDS_KEYS;
    const bool hist = bounded && vocab > SMP_HIST_MIN;
    hipLaunchKernelGGL(k_sample_max, dim3(nb, rows), dim3(256), 0, s, scores, vocab, maxes, flags, kin, hist);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_sample_p, dim3(nb, rows), dim3(256), 0, s, scores, vocab, temperature, maxes, flags, kin, kout,
                       hist, full);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (full)
        for (uint32_t r = 0; r < rows; r++) {
            size_t b = sort_bytes;
            e = rocprim::radix_sort_keys(tmp, b, kin + (size_t)r * vocab, kout + (size_t)r * vocab, vocab, 0, 64, s);
            if (e != hipSuccess) return e;
        }
    hipLaunchKernelGGL(k_sample_pick, dim3(rows), dim3(SMP_THREADS), 0, s, kin, kout, vocab, flags, top_p, seed, step0,
                       ids, hist, full);
    return hipGetLastError();
}

}  // namespace bchip
