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
// by one, and the scan goes on behind it with the new binade's ulp. The total goes over segments
// of 512 tokens composed ahead, a wave each, for a guessed binade (k_sample_segs). For 4 rows of
// 151936 that total takes 54 us of one workgroup a row; scanned token by token it took 180, and
// one lane adding the terms 1190.
//
// Only the kept prefix has to be sorted: a histogram of p by its leading bits bounds it from
// below (k_sample_bound), the tokens above the bound are scattered to their bins' places, and
// runs of bins of about 4096 keys are sorted in LDS, a workgroup each. A row of at most 8192
// tokens is sorted whole by the workgroup that picks. Bound by latency: 4 rows of 151936 take
// 139 us from scores to tokens, 1587 with one lane a row and a whole radix sort.
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

constexpr uint32_t SMP_BINS = 2048;      // by the exponent's and three more bits of p in [0, 1]
constexpr uint32_t SMP_LDS_KEYS = 8192;  // keys a workgroup sorts in LDS; longer rows get the histogram
constexpr uint32_t SMP_BUCKET = 4096;    // places whose bins a workgroup sorts together
constexpr uint32_t SMP_BLOCK = 4096;     // tokens a workgroup of the parallel passes
constexpr int SMP_EPT = 8;               // terms a thread of a chunk: 8192 a chunk
constexpr uint32_t SMP_FRONT = 512;      // sorted candidates whose sums one lane takes

__device__ __forceinline__ uint32_t p_bin(float p) { return min(__float_as_uint(p) >> 19, SMP_BINS - 1u); }  // p in [0, 1]

constexpr uint32_t SMP_SEG = 64 * SMP_EPT;  // tokens a segment of the total: a wave's

// A segment's terms composed for the binade e its sum is guessed to stay in (0: no guess).
struct SmpSeg {
    uint2 c;
    uint32_t e;
    float sum;  // about its sum
};

// A row's histogram, in the half of its sorted keys' space that p (f32) leaves free: mass (2^-40
// units, rounded down), tokens, and the bins' first places, later cursors (from the top bin down).
struct SmpHist {
    uint64_t mass[SMP_BINS];
    uint32_t count[SMP_BINS], place[SMP_BINS];
};
__device__ __forceinline__ SmpHist* hist_of(uint64_t* p_row, uint32_t vocab) {
    return (SmpHist*)(p_row + (vocab - (uint32_t)(sizeof(SmpHist) / sizeof(uint64_t))));
}
static_assert((SMP_LDS_KEYS + 1) * 8 >= (SMP_LDS_KEYS + 1) * 4 + 4 + sizeof(SmpHist), "p and the histogram share a row");

// What the passes of a row leave for each other.
struct SmpRow {
    uint32_t nan;    // a p is NaN
    float total;
    uint32_t bound;  // the lowest bin of the candidates
    uint32_t ncand;
};

// Max of each block of a row; clears the row's histogram and NaN flag.
__global__ __launch_bounds__(256) void k_sample_max(const float* __restrict__ scores, uint32_t vocab,
                                                    float* __restrict__ maxes, SmpRow* __restrict__ info,
                                                    uint64_t* __restrict__ p_out, bool hist) {
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
        if (blockIdx.x == 0) info[row].nan = 0u;
    }
    if (hist) {
        SmpHist* h = hist_of(p_out + (size_t)row * vocab, vocab);
        for (uint32_t i = blockIdx.x * 256 + tid; i < SMP_BINS; i += nb * 256) {
            h->mass[i] = 0;
            h->count[i] = 0;
        }
    }
}

// p of every token (f32, rows vocab u64 apart), and the histogram of the tokens with p > 0.
__global__ __launch_bounds__(256) void k_sample_p(const float* __restrict__ scores, uint32_t vocab, float temperature,
                                                  const float* __restrict__ maxes, SmpRow* __restrict__ info,
                                                  uint64_t* __restrict__ p_out, SmpSeg* __restrict__ segs, uint32_t nseg,
                                                  bool hist) {
    __shared__ uint64_t hm[SMP_BINS];
    __shared__ uint32_t hc[SMP_BINS];
    __shared__ float seg_sum[SMP_BLOCK / SMP_SEG];
    const uint32_t tid = threadIdx.x, row = blockIdx.y, nb = gridDim.x;
    const float* s = scores + (size_t)row * vocab;
    float* pr = (float*)(p_out + (size_t)row * vocab);
    float mx = -INFINITY;
    for (uint32_t i = tid & 63; i < nb; i += 64) mx = fmaxf(mx, maxes[(size_t)row * nb + i]);
#pragma unroll
    for (int d = 1; d < 64; d *= 2) mx = fmaxf(mx, __shfl_xor(mx, d));
    if (hist)
        for (uint32_t i = tid; i < SMP_BINS; i += 256) {
            hm[i] = 0;
            hc[i] = 0;
        }
    if (tid < SMP_BLOCK / SMP_SEG) seg_sum[tid] = 0.0f;
    __syncthreads();
    const uint32_t c0 = blockIdx.x * SMP_BLOCK, c1 = min(c0 + SMP_BLOCK, vocab);
    bool nan = false;
    for (uint32_t i0 = c0; i0 < c1; i0 += 256) {
        const uint32_t i = i0 + tid;
        const float p = i < c1 ? (float)exp((double)((s[i] - mx) / temperature)) : 0.0f;
        nan = nan || isnan(p);
        if (i < c1) pr[i] = p;
        if (hist) {
            if (p > 0.0f) {
                atomicAdd((unsigned long long*)&hm[p_bin(p)], (unsigned long long)(p * 1099511627776.0f));
                atomicAdd(&hc[p_bin(p)], 1u);
            }
            float sum = p;
#pragma unroll
            for (int d = 1; d < 64; d *= 2) sum += __shfl_xor(sum, d);
            if ((tid & 63) == 0) atomicAdd(&seg_sum[(i0 - c0) / SMP_SEG], sum);
        }
    }
    if (nan) info[row].nan = 1u;
    if (hist) {
        __syncthreads();
        const uint32_t seg = blockIdx.x * (SMP_BLOCK / SMP_SEG) + tid;
        if (tid < SMP_BLOCK / SMP_SEG && seg < nseg) segs[(size_t)row * nseg + seg].sum = seg_sum[tid];
        SmpHist* h = hist_of(p_out + (size_t)row * vocab, vocab);
        for (uint32_t i = tid; i < SMP_BINS; i += 256)
            if (hc[i]) {
                atomicAdd((unsigned long long*)&h->mass[i], (unsigned long long)hm[i]);
                atomicAdd(&h->count[i], hc[i]);
            }
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

// A thread's terms in ulps of 2^(e - 150): the mantissa shifted by the exponents' difference k,
// the bits shifted out against one half.
__device__ __forceinline__ uint2 terms(const float (&v)[SMP_EPT], int e) {
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
    if (!ties) return uint2{sum, sum};
    uint2 a = uint2{0u, 0u};
#pragma unroll
    for (int j = 0; j < SMP_EPT; j++)
        a = compose(a, ties >> j & 1u ? uint2{q[j] + (q[j] & 1u), q[j] + 1u - (q[j] & 1u)} : uint2{q[j], q[j]});
    return a;
}

// A sum's binade (biased exponent, at least 1) and its ulps; and back.
__device__ __forceinline__ void split_sum(float s, int& e, uint32_t& m) {
    const uint32_t bits = __float_as_uint(s) & 0x7fffffffu;
    e = (int)max(bits >> 23, 1u);
    m = (bits & 0x7fffffu) | (bits >> 23 ? 0x800000u : 0u);
}
__device__ __forceinline__ float join_sum(int e, uint32_t m) {
    return __uint_as_float(m & 0x800000u ? ((uint32_t)e << 23) | (m & 0x7fffffu) : m);  // (else subnormal: e is 1)
}
// Inclusive composition over the wave's lanes.
__device__ __forceinline__ uint2 wave_compose(uint2 a, uint32_t lane) {
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
        const uint2 o = uint2{__shfl_up(a.x, d), __shfl_up(a.y, d)};
        if (lane >= (uint32_t)d) a = compose(o, a);
    }
    return a;
}

// The serial sum s plus the wave's 64 x SMP_EPT terms (those past the list 0), to every lane:
// run_chunk's additions within a wave.
__device__ float wave_chunk(float s, const float (&v)[SMP_EPT]) {
    const uint32_t lane = threadIdx.x & 63;
    for (uint32_t t0 = 0; t0 < 64;) {
        int e;
        uint32_t m;
        split_sum(s, e, m);
        uint2 a = terms(v, e);
        if (lane < t0) a = uint2{0u, 0u};
        a = wave_compose(a, lane);
        const uint32_t past = m + ((m & 1u) ? a.y : a.x);
        const uint64_t b = __ballot(lane >= t0 && past >= 0x1000000u);
        const float after = join_sum(e, past);
        if (!b) return __shfl(after, 63);
        const uint32_t f = (uint32_t)__builtin_ctzll(b);
        if (f > t0) s = __shfl(after, (int)f - 1);
        float x = s;
#pragma unroll
        for (int j = 0; j < SMP_EPT; j++) x += v[j];
        s = __shfl(x, (int)f);
        t0 = f + 1;
    }
    return s;
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
        int e;
        uint32_t m;
        split_sum(s0, e, m);  // s0 = m ulps of 2^(e - 150)
        uint2 a = terms(v, e);
        if (tid < t0) a = uint2{0u, 0u};
        a = wave_compose(a, lane);
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
        const float after = join_sum(e, past);
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

// Ascending radix sort of n keys by one workgroup through memory (a and b in turn; returns the one
// that holds the result): a bin of more keys than LDS takes, so of nearly equal p.
__device__ uint64_t* radix_sort_keys_wg(uint64_t* a, uint64_t* b, uint32_t n, uint32_t* base, uint32_t (*cnt)[256]) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    for (int sh = 0; sh < 64; sh += 8) {
        if (tid < 256) base[tid] = 0;
        __syncthreads();
        for (uint32_t i = tid; i < n; i += SMP_THREADS) atomicAdd(&base[(a[i] >> sh) & 255u], 1u);
        __syncthreads();
        if (base[(a[0] >> sh) & 255u] == n) {  // one digit for all
            __syncthreads();
            continue;
        }
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
            const uint64_t key = have ? a[i0 + tid] : 0;
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
                b[at] = key;
            }
            __syncthreads();
            if (tid < 256)
                for (uint32_t k = 0; k < SMP_THREADS / 64; k++) base[tid] += cnt[k][tid];
            __syncthreads();
        }
        __threadfence();
        __syncthreads();
        uint64_t* t = a;
        a = b;
        b = t;
    }
    return a;
}

// Ascending sort of ks[0 .. n), n <= SMP_LDS_KEYS, by the workgroup (bitonic, padded with ~0).
__device__ void lds_sort(uint64_t* ks, uint32_t n) {
    const uint32_t tid = threadIdx.x;
    uint32_t np = 1;
    while (np < n) np *= 2;
    for (uint32_t i = n + tid; i < np; i += SMP_THREADS) ks[i] = ~0ull;
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
}

// The same over t[0 .. n) in LDS (n > 0, zeros up to a multiple of 8) by one lane, from start, into
// sc.sum; returns the term's index or -1: for the first few hundred terms, in which a sum leaves a
// binade every few (a binade left costs run_chunk 1.5 us) and a nucleus often ends. 2000 tokens at T
// 0.3, top_p 0.5, 75 -> 42 us, 100 tokens 37 -> 17; 4 rows of 151936 137 -> 103.
template <bool SUB, bool TARGET>
__device__ int run_front(SmpScan& sc, const float* t, uint32_t n, float start, float target) {
    __syncthreads();  // the terms are there
    if (threadIdx.x == 0) {
        float s = start;
        uint32_t found = 0xffffffffu;
        f32x4 a = *(const f32x4*)t, b = *(const f32x4*)(t + 4);
        for (uint32_t i = 0; i < n; i += 8) {
            const float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
            const uint32_t next = min(i + 8, (n - 1) & ~7u);
            a = *(const f32x4*)(t + next);
            b = *(const f32x4*)(t + next + 4);
            float r[8];
#pragma unroll
            for (int j = 0; j < 8; j++) r[j] = SUB ? (j ? r[j - 1] : s) - v[j] : (j ? r[j - 1] : s) + v[j];
            s = r[7];
            if (TARGET && (SUB ? s <= 0.0f : s >= target)) {  // (the sums are monotone)
                int j = 0;
                while (SUB ? r[j] > 0.0f : r[j] < target) j++;
                found = i + (uint32_t)j;
                break;
            }
        }
        sc.sum = s;
        sc.found = found;
    }
    __syncthreads();
    return (int)sc.found;
}

__device__ __forceinline__ void load_terms(const float* p, uint32_t i0, uint32_t vocab, float (&v)[SMP_EPT]) {
#pragma unroll
    for (int j = 0; j < SMP_EPT; j++) v[j] = i0 + j < vocab ? p[i0 + j] : 0.0f;
}

// Each segment's terms composed for the binade that the segments' rough sums put it in, a wave a
// segment; none where those sums leave the binade open. A wrong guess costs time only.
__global__ __launch_bounds__(256) void k_sample_segs(const uint64_t* __restrict__ p_out, uint32_t vocab,
                                                     SmpSeg* __restrict__ segs, uint32_t nseg) {
    const uint32_t lane = threadIdx.x & 63, seg = blockIdx.x * 4 + (threadIdx.x >> 6), row = blockIdx.y;
    if (seg >= nseg) return;
    SmpSeg* sg = segs + (size_t)row * nseg;
    float before = 0.0f;
    for (uint32_t k = lane; k < seg; k += 64) before += sg[k].sum;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) before += __shfl_xor(before, d);
    int e0, e1;
    uint32_t m;
    split_sum(before * 0.999f, e0, m);
    split_sum((before + sg[seg].sum) * 1.001f, e1, m);
    if (e0 != e1 || before == 0.0f) {
        if (lane == 0) sg[seg].e = 0;
        return;
    }
    float v[SMP_EPT];
    load_terms((const float*)(p_out + (size_t)row * vocab), seg * SMP_SEG + lane * SMP_EPT, vocab, v);
    const uint2 a = wave_compose(terms(v, e0), lane);
    if (lane == 63) {
        sg[seg].c = a;
        sg[seg].e = (uint32_t)e0;
    }
}

// The row's serial total from its segments, to every thread: within a binade the segments compose
// as terms do (run_chunk's scan, a segment a thread); one without a right guess, or in which
// the sum leaves its binade, is added by wave 0 (wave_chunk).
__device__ float segment_total(SmpScan& sc, const float* p, uint32_t vocab, const SmpSeg* sg, uint32_t nseg) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (tid == 0) sc.sum = -0.0f;
    for (uint32_t w0 = 0; w0 < nseg; w0 += SMP_THREADS) {
        const uint32_t nw = min((uint32_t)SMP_THREADS, nseg - w0);
        const uint2 mine = tid < nw ? sg[w0 + tid].c : uint2{0u, 0u};
        const uint32_t mine_e = tid < nw ? sg[w0 + tid].e : 0u;
        if (tid == 0) {
            sc.next = 0;
            sc.first[0] = sc.first[1] = 0xffffffffu;
        }
        __syncthreads();
        for (uint32_t turn = 0;; turn ^= 1u) {
            const uint32_t t0 = sc.next;
            int e;
            uint32_t m;
            split_sum(sc.sum, e, m);
            const bool here = tid >= t0 && tid < nw, bad = here && mine_e != (uint32_t)e;
            uint2 a = here && !bad ? mine : uint2{0u, 0u};
            a = wave_compose(a, lane);
            if (lane == 63) sc.wave[w] = a;
            __syncthreads();
            uint2 wt = sc.wave[lane & (SMP_THREADS / 64 - 1)];
#pragma unroll
            for (int d = 1; d < SMP_THREADS / 64; d *= 2) {
                const uint2 o = uint2{__shfl_up(wt.x, d), __shfl_up(wt.y, d)};
                if (lane >= (uint32_t)d) wt = compose(o, wt);
            }
            const uint2 before = uint2{__shfl(wt.x, (int)w - 1), __shfl(wt.y, (int)w - 1)};
            const uint2 upto = w ? compose(before, a) : a;
            const uint32_t past = m + ((m & 1u) ? upto.y : upto.x);
            const uint64_t b = __ballot(bad || (here && past >= 0x1000000u));
            if (b && lane == 0) atomicMin(&sc.first[turn], 64 * w + (uint32_t)__builtin_ctzll(b));
            __syncthreads();
            const uint32_t f = sc.first[turn];
            if (f == 0xffffffffu ? tid == SMP_THREADS - 1 : (f > t0 && tid == f - 1)) sc.sum = join_sum(e, past);
            __syncthreads();
            if (f == 0xffffffffu) break;
            if (w == 0) {
                float v[SMP_EPT];
                load_terms(p, (w0 + f) * SMP_SEG + lane * SMP_EPT, vocab, v);
                const float s = wave_chunk(sc.sum, v);
                if (lane == 0) {
                    sc.sum = s;
                    sc.next = f + 1;
                    sc.first[turn] = 0xffffffffu;
                }
            }
            __syncthreads();
        }
    }
    const float total = sc.sum;
    __syncthreads();
    return total;
}

// A long row's total, the lowest bin of its candidates and every bin's first place. The running
// f32 mass of k shares p / total, each rounded, falls short of their true sum by less than (k +
// 2) 2^-24 of it, so bins whose true mass M of K tokens gives M / total (1 - (K + 2) 2^-24) >=
// top_p hold the whole kept prefix. Tokens of p = 0 move no sum and are never picked past the
// first place (the largest p is 1), so they are left out. The bound's bins hold at least one
// token, the most likely one, as the reference keeps at least one.
// firsts[k]: the first place at or past k SMP_BUCKET at which a bin of the candidates begins (or
// their end).
__global__ __launch_bounds__(SMP_THREADS) void k_sample_bound(uint64_t* p_out, uint32_t vocab, SmpRow* __restrict__ info,
                                                              uint32_t* __restrict__ firsts, uint32_t nfirst,
                                                              const SmpSeg* __restrict__ segs, uint32_t nseg, float top_p) {
    __shared__ SmpScan sc;
    __shared__ uint64_t wm[SMP_THREADS / 64];
    __shared__ uint32_t wc[SMP_THREADS / 64], bound_s;
    constexpr uint32_t BPT = SMP_BINS / SMP_THREADS;
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6, row = blockIdx.x;
    if (info[row].nan) return;
    uint64_t* pr = p_out + (size_t)row * vocab;
    SmpHist* h = hist_of(pr, vocab);
    const float total = segment_total(sc, (const float*)pr, vocab, segs + (size_t)row * nseg, nseg);
    uint64_t bm[BPT], mass = 0;  // thread t: bins from the top down
    uint32_t bc[BPT], count = 0;
#pragma unroll
    for (uint32_t k = 0; k < BPT; k++) {
        const uint32_t bin = SMP_BINS - 1u - (BPT * tid + k);
        mass += bm[k] = h->mass[bin];
        count += bc[k] = h->count[bin];
    }
    uint64_t rm = mass;
    uint32_t rc = count;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
        const uint64_t om = (uint64_t)__shfl_up((unsigned long long)rm, d);
        const uint32_t oc = __shfl_up(rc, d);
        if (lane >= (uint32_t)d) {
            rm += om;
            rc += oc;
        }
    }
    if (lane == 63) {
        wm[w] = rm;
        wc[w] = rc;
    }
    if (tid == 0) bound_s = 0u;
    __syncthreads();
    for (uint32_t k = 0; k < w; k++) {
        rm += wm[k];
        rc += wc[k];
    }
    rm -= mass;
    rc -= count;
#pragma unroll
    for (uint32_t k = 0; k < BPT; k++) {
        const uint32_t bin = SMP_BINS - 1u - (BPT * tid + k);
        h->place[bin] = rc;
        rm += bm[k];
        rc += bc[k];
        // (A bin above every token is no bound: at a top_p of 0 or less its mass of 0 would reach it.)
        if (rc > 0 &&
            (double)rm * 9.094947017729282e-13 / (double)total * (1.0 - (double)(rc + 2u) * 5.960464477539063e-8) >= (double)top_p)
            atomicMax(&bound_s, bin);
    }
    __syncthreads();
    if (bound_s / BPT == (SMP_BINS - 1u) / BPT - tid) {  // the thread of the bound's bin
        uint32_t upto = rc - count;
#pragma unroll
        for (uint32_t k = 0; k < BPT; k++)
            if (SMP_BINS - 1u - (BPT * tid + k) >= bound_s) upto += bc[k];
        info[row].total = total;
        info[row].bound = bound_s;
        info[row].ncand = upto;
    }
    uint32_t begin = rc - count;
    if (tid == 0) firsts[(size_t)row * nfirst] = 0;
#pragma unroll
    for (uint32_t k = 0; k < BPT; k++) {
        if (SMP_BINS - 1u - (BPT * tid + k) < bound_s) break;
        const uint32_t end = begin + bc[k];
        for (uint32_t f = begin / SMP_BUCKET + 1; f * SMP_BUCKET <= end; f++) firsts[(size_t)row * nfirst + f] = end;
        begin = end;
    }
}

// The candidates' keys to their bins' places (in any order within a bin: k_sample_sort follows).
__global__ __launch_bounds__(256) void k_sample_scatter(uint64_t* __restrict__ p_out, uint32_t vocab,
                                                        const SmpRow* __restrict__ info, uint64_t* __restrict__ keys) {
    const uint32_t row = blockIdx.y;
    if (info[row].nan) return;
    const uint32_t bound = info[row].bound;
    uint64_t* pr = p_out + (size_t)row * vocab;
    const float* p = (const float*)pr;
    SmpHist* h = hist_of(pr, vocab);
    const uint32_t c0 = blockIdx.x * SMP_BLOCK, c1 = min(c0 + SMP_BLOCK, vocab);
    for (uint32_t i = c0 + threadIdx.x; i < c1; i += 256) {
        const float x = p[i];
        if (x > 0.0f && p_bin(x) >= bound) keys[(size_t)row * vocab + atomicAdd(&h->place[p_bin(x)], 1u)] = sort_key(x, i);
    }
}

// Workgroup (k, row) sorts the candidates of the bins that begin in places [k, k + 1) SMP_BUCKET.
// (spare: p's and the histogram's space, no longer needed.)
__global__ __launch_bounds__(SMP_THREADS) void k_sample_sort(uint32_t vocab, const SmpRow* __restrict__ info,
                                                             const uint32_t* __restrict__ firsts, uint32_t nfirst,
                                                             uint64_t* __restrict__ keys, uint64_t* __restrict__ spare) {
    __shared__ uint64_t ks[SMP_LDS_KEYS];
    __shared__ uint32_t cnt[SMP_THREADS / 64][256], base[256];
    const uint32_t tid = threadIdx.x, row = blockIdx.y, k = blockIdx.x;
    if (info[row].nan || k * SMP_BUCKET >= info[row].ncand) return;
    const uint32_t* f = firsts + (size_t)row * nfirst + k;
    const uint32_t lo = f[0], hi = (k + 1) * SMP_BUCKET <= info[row].ncand ? f[1] : info[row].ncand;
    if (lo >= hi) return;
    uint64_t* kr = keys + (size_t)row * vocab + lo;
    const uint32_t n = hi - lo;
    if (n <= SMP_LDS_KEYS) {
        for (uint32_t i = tid; i < n; i += SMP_THREADS) ks[i] = kr[i];
        __syncthreads();
        lds_sort(ks, n);
        for (uint32_t i = tid; i < n; i += SMP_THREADS) kr[i] = ks[i];
    } else {
        uint64_t* other = spare + (size_t)row * vocab + lo;
        const uint64_t* got = radix_sort_keys_wg(kr, other, n, base, cnt);
        if (got != kr)
            for (uint32_t i = tid; i < n; i += SMP_THREADS) kr[i] = got[i];
    }
}

// Per row: the nucleus and the draw over the sorted candidates (hist: keys, sorted; else the
// whole row's p, sorted here).
__global__ __launch_bounds__(SMP_THREADS) void k_sample_pick(const uint64_t* __restrict__ keys,
                                                             const uint64_t* __restrict__ p_out, uint32_t vocab,
                                                             const SmpRow* __restrict__ info, float top_p, uint64_t seed,
                                                             uint64_t step0, uint32_t* __restrict__ ids, bool hist) {
    __shared__ SmpScan sc;
    __shared__ __attribute__((aligned(16))) uint64_t ks[SMP_LDS_KEYS];
    __shared__ __attribute__((aligned(16))) float fp[SMP_FRONT], fs[SMP_FRONT];  // the first candidates' p and shares
    __shared__ uint64_t best[SMP_THREADS / 64];
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6, row = blockIdx.x;
    const uint64_t* kr = keys + (size_t)row * vocab;
    const float* pr = (const float*)(p_out + (size_t)row * vocab);
    if (info[row].nan) {
        // A NaN: total and every running mass are NaN, nothing is reached, and the pick is the first
        // of the order.
        uint64_t k = ~0ull;
        for (uint32_t i = tid; i < vocab; i += SMP_THREADS) k = min(k, sort_key(pr[i], i));
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
    float total;
    uint32_t ncand;
    if (hist) {
        total = info[row].total;
        ncand = info[row].ncand;
    } else {
        float* t = (float*)ks;
        for (uint32_t i = tid; i < (vocab + 7) / 8 * 8; i += SMP_THREADS) t[i] = i < vocab ? pr[i] : 0.0f;
        // (8192 tokens 105 us, 141 by one lane; 2000 42, 45 with a chunk and up to 98 where the scores ascend)
        const uint32_t tf = vocab <= 4096 ? vocab : 2 * SMP_FRONT;
        run_front<false, false>(sc, t, tf, -0.0f, 0.0f);
        if (tf < vocab) {  // (one chunk: at most SMP_LDS_KEYS terms)
            float v[SMP_EPT];
            const uint32_t i0 = tf + tid * SMP_EPT;
            load_terms(t, i0, vocab, v);
            run_chunk<false, false>(sc, v, i0 < vocab ? (int)min((uint32_t)SMP_EPT, vocab - i0) : 0, 0.0f);
        }
        total = sc.sum;
        ncand = vocab;
        __syncthreads();
        for (uint32_t i = tid; i < vocab; i += SMP_THREADS) ks[i] = sort_key(pr[i], i);
        __syncthreads();
        lds_sort(ks, vocab);
    }
    auto key_at = [&](uint32_t i) { return hist ? kr[i] : ks[i]; };
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
    const uint32_t nf = min(ncand, SMP_FRONT);
    for (uint32_t i = tid; i < (nf + 7) / 8 * 8; i += SMP_THREADS) {
        const float p = i < nf ? key_weight(key_at(i)) : 0.0f;
        fp[i] = p;
        fs[i] = i < nf ? p / total : 0.0f;
    }
    // keep: the running mass reaches top_p.
    uint32_t keep = ncand;
    int at = run_front<false, true>(sc, fs, nf, 0.0f, top_p);
    if (at >= 0) keep = (uint32_t)at + 1;
    for (uint32_t c0 = nf; c0 < ncand && at < 0; c0 += SMP_THREADS * SMP_EPT) {
        float v[SMP_EPT];
        const int n = load(c0, ncand, v, true);
        at = run_chunk<false, true>(sc, v, n, top_p);
        if (at >= 0) keep = c0 + (uint32_t)at + 1;
    }
    // The kept mass, in sorted order from -0, and the draw (zeros behind the kept ones).
    const uint32_t kf = min(keep, nf);
    __syncthreads();
    for (uint32_t i = kf + tid; i < (kf + 7) / 8 * 8; i += SMP_THREADS) fp[i] = 0.0f;
    run_front<false, false>(sc, fp, kf, -0.0f, 0.0f);
    for (uint32_t c0 = kf; c0 < keep; c0 += SMP_THREADS * SMP_EPT) {
        float v[SMP_EPT];
        const int n = load(c0, keep, v, false);
        run_chunk<false, false>(sc, v, n, 0.0f);
    }
    const float kept = sc.sum;
    const uint64_t step = step0 + row;
    uint32_t id = (uint32_t)(key_at(0) & 0xffffffffu);
    at = run_front<true, true>(sc, fp, kf, uniform(seed ^ (step * 0x9e3779b97f4a7c15ull)) * kept, 0.0f);
    if (at >= 0) id = (uint32_t)(key_at((uint32_t)at) & 0xffffffffu);
    for (uint32_t c0 = kf; c0 < keep && at < 0; c0 += SMP_THREADS * SMP_EPT) {
        float v[SMP_EPT];
        const int n = load(c0, keep, v, false);
        at = run_chunk<true, true>(sc, v, n, 0.0f);
        if (at >= 0) id = (uint32_t)(key_at(c0 + (uint32_t)at) & 0xffffffffu);
    }
    if (tid == 0) ids[row] = id;
}

static uint32_t sample_blocks(uint32_t vocab) { return (vocab + SMP_BLOCK - 1) / SMP_BLOCK; }

static uint32_t sample_segs(uint32_t vocab) { return (vocab + SMP_SEG - 1) / SMP_SEG; }
static uint32_t sample_firsts(uint32_t vocab) { return vocab / SMP_BUCKET + 2; }

// Keys twice (the second also holds p and the histogram), the segments, the rows' facts, the
// blocks' maxima and the buckets.
size_t sample_scratch_bytes(uint32_t rows, uint32_t vocab) {
    return (size_t)rows * (2 * (size_t)vocab * sizeof(uint64_t) + sizeof(SmpRow) + sample_blocks(vocab) * sizeof(float) +
                          sample_firsts(vocab) * sizeof(uint32_t) + sample_segs(vocab) * sizeof(SmpSeg)) + 512;
}

hipError_t sample_launch(const float* scores, uint32_t rows, uint32_t vocab, float temperature, float top_p,
                         uint64_t seed, uint64_t step0, uint32_t* ids, void* scratch, size_t scratch_bytes,
                         hipStream_t s) {
    if (rows == 0 || vocab == 0) return hipSuccess;
    if (!(temperature > 0.0f)) {
        hipLaunchKernelGGL(k_argmax, dim3(rows), dim3(SMP_THREADS), 0, s, scores, vocab, ids);
        return hipGetLastError();
    }
    if (scratch_bytes < sample_scratch_bytes(rows, vocab)) return hipErrorInvalidValue;
    const uint32_t nb = sample_blocks(vocab);
    uint64_t* keys = (uint64_t*)(((uintptr_t)scratch + 255) & ~(uintptr_t)255);
    uint64_t* p_out = keys + (size_t)rows * vocab;
    SmpSeg* segs = (SmpSeg*)(((uintptr_t)(p_out + (size_t)rows * vocab) + 15) & ~(uintptr_t)15);
    const uint32_t nseg = sample_segs(vocab);
    SmpRow* info = (SmpRow*)(segs + (size_t)rows * nseg);
    float* maxes = (float*)(info + rows);
    uint32_t* firsts = (uint32_t*)(maxes + (size_t)rows * nb);
    const uint32_t nfirst = sample_firsts(vocab);
    const bool hist = vocab > SMP_LDS_KEYS;
    hipLaunchKernelGGL(k_sample_max, dim3(nb, rows), dim3(256), 0, s, scores, vocab, maxes, info, p_out, hist);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_sample_p, dim3(nb, rows), dim3(256), 0, s, scores, vocab, temperature, maxes, info, p_out,
                       segs, nseg, hist);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (hist) {
        hipLaunchKernelGGL(k_sample_segs, dim3((nseg + 3) / 4, rows), dim3(256), 0, s, p_out, vocab, segs, nseg);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_sample_bound, dim3(rows), dim3(SMP_THREADS), 0, s, p_out, vocab, info, firsts,
                           nfirst, segs, nseg, top_p);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_sample_scatter, dim3(nb, rows), dim3(256), 0, s, p_out, vocab, info, keys);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_sample_sort, dim3((vocab + SMP_BUCKET - 1) / SMP_BUCKET, rows), dim3(SMP_THREADS), 0, s, vocab,
                           info, firsts, nfirst, keys, p_out);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_sample_pick, dim3(rows), dim3(SMP_THREADS), 0, s, keys, p_out, vocab, info, top_p, seed, step0,
                       ids, hist);
    return hipGetLastError();
}

}  // namespace bchip
