// Attention over an f32 cache in f32 arithmetic: the path for callers that keep bc-infer's
// own f32 cache (crates/bc-infer/src/gpu/mod.rs:409-421) and want its results to f32
// rounding, as the reference's end-to-end tests demand (model.rs:531, 548, 642: 1e-4).
//
// The reference per (row, head) (model.rs:448-481): scores dot(q, k) * scale, one softmax over
// the whole list, then o += (p / sum) v in slot order. Here both contractions run on the f32
// matrix cores (v_mfma_f32_16x16x4_f32: f32 operands, products and sums): a dot as eight chains of
// hd / 8 products, added in pairs, times scale * log2(e); the softmax is online, over blocks of
// F32_BLK list entries in exp2 units: per block and slot, the block's max, the new running
// max, P = 2^(s - max), the block's sum of P and of P v (a chain over its entries), and
// the running state scaled by 2^(old max - new max). Lists go in chunks of CHUNK_MULTI
// entries, each an online softmax from a fresh state, folded left to right (merge_coef, the
// fold every other kernel and attn_combine use). A row's bits therefore depend only on its q
// and its list: the same in any batch, as a tree node or a line token, split over
// workgroups or not, and a one-row pass gives the bits of the same row in a batch.
//
// A tile is 16 query slots of one KV head (rows x heads of the group; one row of a tree). S^T =
// K Q^T leaves entry 4 (l / 16) + i of a 16-entry tile and slot l % 16 in lane l, register i,
// which is the second product's operand (O^T = V^T P^T) as it stands: no move between lanes,
// and a slot's max, sum and scale sit in the lanes that hold its outputs. The contractions' order
// within a step of four is free (dims 16 j + 4 g + c, entries 4 g + i for lane group g = l / 16),
// so that every operand is a 16-byte read.
//
// Two forms, the same bits. attn_f32_step: a workgroup per (tile, chunk), its waves each three
// of the chunk's 16-entry score tiles and a quarter of the output dims; K and V go straight to
// registers, a chunk's K all in flight at once. attn_f32_line: a workgroup of four
// tiles walks the whole list, K and V blocks staged in LDS for all four.
#include "common.hpp"
#include "internal.hpp"

#include <hip/hip_ext.h>
#include <math.h>

#include <type_traits>

namespace bchip {

constexpr int F32_BLK = 32;      // list entries per block
constexpr int F32_SLOTS = 16;    // query slots a tile
constexpr int F32_THREADS = 256;
constexpr int F32_WAVES = F32_THREADS / 64;

struct F32Params {
    const float* q;
    const float* kc;  // the row's cache (a ragged pool's offset applied)
    const float* vc;
    float* out;
    float* part_o;    // [unit][F32_SLOTS][HD]: chunk states of split launches
    float* part_ml;   // [unit][F32_SLOTS][2]
    const uint32_t* masks;
    uint32_t tree;
    uint32_t rows, nh, nkv, hd, G;
    uint32_t pos;     // line: slot of row 0; tree: the tree's first slot
    uint64_t slot_limit;  // slots the caches hold (tree slots past it read as zeros)
    float sc;         // scale * log2(e)
    uint32_t rb, nrb; // rows a tile (1 for trees), tiles of a KV head
    // A split tree's chunks wholly below pos, which hold the same slots for every row: chunks,
    // rows a tile, tiles of a KV head (npc 0: none such).
    uint32_t npc, prb, npt;
    uint32_t nchunk;  // chunks of the farthest list
    uint32_t split;   // attn_f32_step: more than one chunk, the states go to attn_combine
    const float* zero;  // ZERO_BYTES of zeros: the loads of rows past a list
    // A line call fused with RoPE and the K/V append of its rows at slots pos .. pos + rows - 1
    // (attn_f32_step's NR > 0: at most NR rows): q is unrotated on entry and rotated as it
    // is staged; the new K rows (knew, rotated here) and V rows (vnew) go to the caches and
    // stand in for those slots' cache entries. q is left rotated: by the workgroup itself when
    // unsplit, else by the fold.
    const float* knew;
    const float* vnew;
    const float* inv_freq;
    const uint32_t* positions;  // positions[r]: row r's rotation position
    uint32_t rope_dim, neox;
    float* qw;
};

// Rows a fused line call of several rows takes.
constexpr uint32_t F32_FUSE_ROWS = 8;

// Lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and D[4 (l / 16) + i][l % 16].
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The max of a slot's four lanes (l, l ^ 16, l ^ 32, l ^ 48), to each of them; their sum.
__device__ __forceinline__ float slot_max(float x) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float slot_sum(float x) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// A score tile from its eight chains: entries first .. first + 3 of the list in a lane; -inf at
// or past the slot's list.
__device__ __forceinline__ f32x4 score_tile(const f32x4 (&a)[8], float sc, uint32_t first, uint32_t len) {
    f32x4 s;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float d = ((a[0][i] + a[1][i]) + (a[2][i] + a[3][i])) + ((a[4][i] + a[5][i]) + (a[6][i] + a[7][i]));
        s[i] = first + i < len ? d * sc : -INFINITY;
    }
    return s;
}

// A slot's running max and this lane's share of its sum, taken over a block: s becomes P; returns
// the scale of what came before.
__device__ __forceinline__ float softmax_block(f32x4 (&s)[2], float& m, float& l) {
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; t++) mx = fmaxf(mx, fmaxf(fmaxf(s[t][0], s[t][1]), fmaxf(s[t][2], s[t][3])));
    const float mn = fmaxf(m, slot_max(mx)), ms = (mn == -INFINITY) ? 0.0f : mn;
    const float cr = exp2_hw(m - ms);
    float bl[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
#pragma unroll
        for (int i = 0; i < 4; i++) s[t][i] = exp2_hw(s[t][i] - ms);
        bl[t] = (s[t][0] + s[t][1]) + (s[t][2] + s[t][3]);
    }
    l = l * cr + (bl[0] + bl[1]);
    m = mn;
    return cr;
}

typedef __amdgpu_buffer_rsrc_t f32_rsrc;

template <int N>
struct VecN {
    typedef float T __attribute__((ext_vector_type(N)));
};
template <>
struct VecN<1> {
    typedef float T;
};
__device__ __forceinline__ float vec_at(float v, int) { return v; }
template <typename V>
__device__ __forceinline__ float vec_at(V v, int i) {
    return v[i];
}

// Bound: HBM for long lists (llama-8B heads, 32768 slots: 268 MB in 59 us a layer, 67 with VALU
// dots; 6001 slots 14.5 against 19), else the fixed time of a launch. K goes out first and V as
// K's registers free up, a third after each score tile: with V's loads queued beside K's the
// first scores came later and the products after them were not hidden (12000 slots: 8 layers
// 255 us, so 237). Steps and verify rows run best two workgroups a CU with these registers;
// trees and short prompts, whose rows read one prefix from cache, three (33 rows at 3001: 265
// us, 236).
// SHORT: lists of at most F32_SHORT entries skip the loads of blocks past them, which take their time
// although they fetch nothing (one row at 0 slots, llama-8B heads, 6.8 -> 4.9 us, at 50 7.8 -> 5.7,
// a tree of 4 rows at 0 8.6 -> 4.9); in longer lists the branches cost 2-10% (6000 slots 19.1 -> 20.4).
template <int HD, int NR, bool SHORT>
__global__ __launch_bounds__(F32_THREADS, HD > 128 ? 1 : NR == 0 ? 3 : 2) void attn_f32_step(const F32Params p) {
    constexpr bool FUSE = NR > 0;
    constexpr int NJ = HD / 16;                      // 16-byte reads of a K row a lane
    constexpr int QS = HD + 4;                       // LDS row of q
    constexpr int NT = CHUNK_MULTI / 16;             // score tiles of a chunk
    constexpr int TPW = NT / F32_WAVES;              // of a wave
    constexpr int VW = HD >= 64 ? HD / F32_WAVES : 16;  // output dims of a wave (hd 32: of two waves)
    constexpr int VC = VW / 16;                      // tiles of them: dim VW w + VC m + c is row m of tile c
    static_assert(NT % F32_WAVES == 0 && F32_BLK == 32, "");
    typedef typename VecN<VC>::T vvec;
    __shared__ __attribute__((aligned(16))) float qs[F32_SLOTS][QS];
    __shared__ __attribute__((aligned(16))) f32x4 ss[NT][64];
    __shared__ uint32_t tail[MAX_ITEMS];
    // FUSE: the new K rows (rotated) and V rows as the caches hold them.
    __shared__ __attribute__((aligned(16))) float nrow[FUSE ? 2 : 1][FUSE ? NR : 1][FUSE ? HD : 4];

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t n = lane & 15u, g = lane >> 4;    // n: an entry, a slot or a dim's place
    // The tiles of a chunk of a KV head side by side in launch order, so that they find its K and V
    // in cache.
    const uint32_t kvh = blockIdx.x % p.nkv, b0 = blockIdx.x / p.nkv, np = p.npc * p.npt;
    const bool prefix = !FUSE && b0 < np;  // a tree's rows together
    const uint32_t rb = prefix ? p.prb : p.rb;
    const uint32_t rbi = prefix ? b0 % p.npt : (b0 - np) % p.nrb, c = prefix ? b0 / p.npt : p.npc + (b0 - np) / p.nrb;
    const uint32_t r0 = rbi * rb, hd = p.hd, kvd = p.nkv * hd;
    const bool tree = p.tree && !prefix;

    // Else a tree's tile is one row: its list is the slots below pos, then pos + j for each set bit j
    // of its mask, in order (kernels.h:266-278).
    uint32_t ntail = 0;
    if (tree) {
        const uint32_t lo = p.masks[2 * r0], hi = p.masks[2 * r0 + 1];
        ntail = __popc(lo) + __popc(hi);
        if (tid < ntail) tail[tid] = p.pos + nth_set_bit(lo, hi, tid);
        __syncthreads();
    }
    // Slot n: head kvh * G + n / rb of row r0 + n % rb.
    auto slot_valid = [&](uint32_t k) { return k / rb < p.G && r0 + k % rb < p.rows; };
    const uint32_t rlast = min(r0 + rb, p.rows) - 1u;
    const uint32_t maxlen = p.tree ? p.pos + ntail : p.pos + rlast + 1u;
    const uint32_t len = !slot_valid(n) ? 0u : p.tree ? maxlen : p.pos + r0 + n % rb + 1u;
    const uint32_t kb0 = c * CHUNK_MULTI, kb1 = min(kb0 + CHUNK_MULTI, maxlen);

    // K and V through buffer descriptors from the chunk's first slot on: entries past the list and
    // dims past hd are sent past the end, as slots past the cache are, and read as 0. (A list's
    // slots lie at most MAX_ITEMS past its entries' numbers.)
    const uint64_t slots = p.slot_limit > kb0 ? min(p.slot_limit - kb0, (uint64_t)(CHUNK_MULTI + MAX_ITEMS)) : 0;
    const size_t at = ((size_t)kb0 * p.nkv + kvh) * hd;
    const int bytes = slots ? (int)((slots * kvd - (size_t)kvh * hd) * 4) : 0;
    const f32_rsrc kr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.kc + at), 0, bytes, 0x00020000);
    const f32_rsrc vr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.vc + at), 0, bytes, 0x00020000);
    constexpr uint32_t NONE = 0x80000000u;
    auto row_at = [&](uint32_t e) -> uint32_t {  // bytes from the chunk's first slot to entry e
        const uint32_t kk = kb0 + e;
        uint32_t s = e;
        if (tree && kk >= p.pos) s = tail[min(kk - p.pos, (uint32_t)MAX_ITEMS - 1u)] - kb0;
        return kk < kb1 ? s * kvd * 4u : NONE;
    };
    const uint32_t nblk = kb0 < kb1 ? (kb1 - kb0 + F32_BLK - 1) / F32_BLK : 0u;
    f32x4 kx[TPW][NJ];
#pragma unroll
    for (int t = 0; t < TPW; t++) {
        if (SHORT && (wave + F32_WAVES * t) / 2 >= nblk) break;
        const uint32_t ro = row_at(16u * (wave + F32_WAVES * t) + n) + 16u * g;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const uint32_t o = (hd == (uint32_t)HD || 16u * j + 4u * g < hd) ? ro + 64u * j : NONE;
            kx[t][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(kr, o, 0, 0));
        }
    }
    const uint32_t vd = VW * wave + VC * n;
    vvec vx[NT][4];
    auto load_v = [&](int t) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t ro = row_at(16u * t + 4u * g + i), o = vd < hd ? ro + 4u * vd : NONE;
            if constexpr (VC == 1)
                vx[t][i] = __builtin_bit_cast(vvec, __builtin_amdgcn_raw_buffer_load_b32(vr, o, 0, 0));
            else if constexpr (VC == 2)
                vx[t][i] = __builtin_bit_cast(vvec, __builtin_amdgcn_raw_buffer_load_b64(vr, o, 0, 0));
            else
                vx[t][i] = __builtin_bit_cast(vvec, __builtin_amdgcn_raw_buffer_load_b128(vr, o, 0, 0));
        }
    };
    const bool has_new = FUSE && kb1 > p.pos && kb0 < p.pos + p.rows;  // a new row's slot is in this chunk
    if constexpr (FUSE) {
        // Row j's new slot is pos + j, its angles from positions[j]; pair pp of a head is (a, b)
        // by rope_pair, rotated when pp < rope_dim / 2 by k_rope_append's expressions (the
        // same bits).
        const uint32_t lo = max(kb0, p.pos), hi = min(kb0 + CHUNK_MULTI, p.pos + p.rows);
        if (lo < hi) {
            // This workgroup reads new slots lo .. hi - 1: their K rows rotated and V rows, into
            // the caches and nrow (tiles of the same chunk write the same values).
            for (uint32_t e = tid; e < (hi - lo) * (HD / 2); e += F32_THREADS) {
                const uint32_t j = lo - p.pos + e / (HD / 2), pp = e % (HD / 2);
                uint32_t a, b;
                const bool rot = rope_pair(pp, p.rope_dim, p.neox, a, b);
                float k0 = 0.0f, k1 = 0.0f, v0 = 0.0f, v1 = 0.0f;
                if (pp < hd / 2) {
                    const float* kn = p.knew + ((size_t)j * p.nkv + kvh) * hd;
                    const float* vn = p.vnew + ((size_t)j * p.nkv + kvh) * hd;
                    k0 = kn[a];
                    k1 = kn[b];
                    if (rot) rotate(kn[a], kn[b], (float)p.positions[j] * p.inv_freq[pp], k0, k1);
                    v0 = vn[2 * pp];
                    v1 = vn[2 * pp + 1];
                    float* kdst = (float*)p.kc + (size_t)(p.pos + j) * kvd + (size_t)kvh * hd;
                    float* vdst = (float*)p.vc + (size_t)(p.pos + j) * kvd + (size_t)kvh * hd;
                    kdst[a] = k0;
                    kdst[b] = k1;
                    vdst[2 * pp] = v0;
                    vdst[2 * pp + 1] = v1;
                }
                nrow[0][j][a] = k0;
                nrow[0][j][b] = k1;
                nrow[1][j][2 * pp] = v0;
                nrow[1][j][2 * pp + 1] = v1;
            }
        }
        // q rotated as it is staged, a pair a thread (dims past hd and empty slots: zeros).
        for (uint32_t e = tid; e < F32_SLOTS * (HD / 2); e += F32_THREADS) {
            const uint32_t k = e / (HD / 2), pp = e % (HD / 2);
            uint32_t a, b;
            const bool rot = rope_pair(pp, p.rope_dim, p.neox, a, b);
            float y0 = 0.0f, y1 = 0.0f;
            if (pp < hd / 2 && slot_valid(k)) {
                const uint32_t r = r0 + k % rb, h = kvh * p.G + k / rb;
                const float* qh = p.q + ((size_t)r * p.nh + h) * hd;
                y0 = qh[a];
                y1 = qh[b];
                if (rot) rotate(qh[a], qh[b], (float)p.positions[r] * p.inv_freq[pp], y0, y1);
            }
            qs[k][a] = y0;
            qs[k][b] = y1;
        }
    } else {
        for (uint32_t e = tid; e < F32_SLOTS * (HD / 4); e += F32_THREADS) {
            const uint32_t k = e / (HD / 4), d = 4 * (e % (HD / 4));
            f32x4 v = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (d < hd && slot_valid(k)) {
                const uint32_t r = r0 + k % rb, h = kvh * p.G + k / rb;
                v = *(const f32x4*)&p.q[((size_t)r * p.nh + h) * hd + d];
            }
            *(f32x4*)&qs[k][d] = v;
        }
    }
    // The fences order LDS only: __syncthreads' would also wait for the K and V loads.
    auto lds_barrier = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    lds_barrier();
    if constexpr (FUSE) {
        if (!p.split) {
            // q stays rotated, as k_rope_append leaves it: this workgroup is the only reader of
            // its heads, and every read of them is done at the barrier. (A split launch's fold
            // writes them once every chunk's workgroup has read them.)
            for (uint32_t e = tid; e < F32_SLOTS * HD; e += F32_THREADS) {
                const uint32_t k = e / HD, d = e % HD;
                if (d < hd && slot_valid(k)) {
                    const uint32_t r = r0 + k % rb, h = kvh * p.G + k / rb;
                    p.qw[((size_t)r * p.nh + h) * hd + d] = qs[k][d];
                }
            }
        }
    }
    f32x4 qx[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) qx[j] = *(const f32x4*)&qs[n][16 * j + 4 * g];

#pragma unroll
    for (int t = 0; t < TPW; t++) {
        const uint32_t tile = wave + F32_WAVES * t, e = kb0 + 16 * tile + n;
        if constexpr (FUSE) {
            // A new row's slot: its K as this kernel wrote it to the cache.
            if (has_new && e >= p.pos && e < p.pos + p.rows) {
#pragma unroll
                for (int j = 0; j < NJ; j++) kx[t][j] = *(const f32x4*)&nrow[0][e - p.pos][16 * j + 4 * g];
            }
        }
        if (tile / 2 < nblk) {
            f32x4 a[8] = {};
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int k = 0; k < 4; k++) a[4 * (j % 2) + k] = mfma4(kx[t][j][k], qx[j][k], a[4 * (j % 2) + k]);
            ss[tile][lane] = score_tile(a, p.sc, kb0 + 16 * tile + 4 * g, len);
        }
#pragma unroll
        for (int v = 0; v < NT / TPW; v++)
            if (!SHORT || (NT / TPW * t + v) / 2u < nblk) load_v(NT / TPW * t + v);
    }
    lds_barrier();

    float m = -INFINITY, l = 0.0f;
    f32x4 o[VC];
#pragma unroll
    for (int k = 0; k < VC; k++) o[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int b = 0; b < NT / 2; b++) {
        if ((uint32_t)b >= nblk) break;
        f32x4 s[2] = {ss[2 * b][lane], ss[2 * b + 1][lane]};
        const float cr = softmax_block(s, m, l);
        f32x4 acc[VC] = {};
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                vvec v = vx[2 * b + t][i];
                if constexpr (FUSE) {
                    const uint32_t e = kb0 + 16 * (2 * b + t) + 4 * g + i;
                    if (has_new && e >= p.pos && e < p.pos + p.rows && vd < (uint32_t)HD)
                        v = *(const vvec*)&nrow[1][e - p.pos][vd];
                }
#pragma unroll
                for (int k = 0; k < VC; k++) acc[k] = mfma4(vec_at(v, k), s[t][i], acc[k]);
            }
#pragma unroll
        for (int k = 0; k < VC; k++)
#pragma unroll
            for (int i = 0; i < 4; i++) o[k][i] = __builtin_fmaf(o[k][i], cr, acc[k][i]);
    }
    l = slot_sum(l);
    // Lane (n, g): dims vb .. vb + 4 VC - 1 of slot n, dim vb + VC i + k in o[k][i].
    const uint32_t vb = VW * wave + 4 * VC * g;
    if (p.split) {
        // A tree's states are its rows' (head n / rb of row r0 + n % rb), a line's its tiles'.
        const size_t u = ((size_t)kvh * p.nrb + (p.tree ? r0 + n % rb : rbi)) * p.nchunk + c;
        const uint32_t at = p.tree ? n / rb : n;
        if (n >= min((uint32_t)F32_SLOTS, p.G * rb) || (prefix && !slot_valid(n))) return;  // attn_combine reads no slot past them
        if (vb < (uint32_t)HD) {
            float* dst = p.part_o + (u * F32_SLOTS + at) * HD + vb;
#pragma unroll
            for (int q4 = 0; q4 < VC; q4++) {
                f32x4 v;
#pragma unroll
                for (int x = 0; x < 4; x++) v[x] = o[(4 * q4 + x) % VC][(4 * q4 + x) / VC];
                *(f32x4*)(dst + 4 * q4) = v;
            }
        }
        if (wave == 0 && g == 0) *(float2*)(p.part_ml + (u * F32_SLOTS + at) * 2) = float2{m, l};
        return;
    }
    if (!slot_valid(n)) return;
    float* dst = p.out + ((size_t)(r0 + n % rb) * p.nh + kvh * p.G + n / rb) * hd + vb;
#pragma unroll
    for (int q4 = 0; q4 < VC; q4++)
        if (vb + 4 * q4 < hd) {
            f32x4 v;
#pragma unroll
            for (int x = 0; x < 4; x++) v[x] = o[(4 * q4 + x) % VC][(4 * q4 + x) / VC] / l;
            *(f32x4*)(dst + 4 * q4) = v;
        }
}

// A block of K or V in LDS, 16-byte units: K's unit u of entry e at u ^ (e % 8), so that the eight
// entries LDS serves together are in eight groups of banks; V's in order. The last V row is zeros:
// what a wave reads for the entries past its tile's lists (another tile's, whose V may be
// infinite or NaN, which a P of 0 would not silence).
template <int HD>
struct F32Stage {
    f32x4 k[F32_BLK][HD / 4];
    f32x4 v[F32_BLK + 1][HD / 4];
};

// Bound: the matrix cores (777 rows at 300, llama-8B heads: 8.8 GFLOP in 127 us, 361 with VALU
// dots; 57 at the rate of a large f32 product). A block's products take 4096 cycles of a
// SIMD at hd 128, so one barrier a block and two workgroups a CU hide the loads. What is left
// is the tail: 392 workgroups of unequal lists over 256 CUs.
// TREE: a row's list by its mask, a tile (one row) a workgroup: only slots too wide for
// attn_f32_step come here.
template <int HD, bool TREE>
__global__ __launch_bounds__(F32_THREADS, HD <= 128 ? 2 : 1) void attn_f32_line(const F32Params p) {
    constexpr int NJ = HD / 16;
    constexpr int VC = HD >= 64 ? 4 : HD / 16;       // a dims tile's lanes are VC dims apart
    constexpr int NH = HD / (16 * VC);               // dim 16 VC h + VC m + c is row m of tile (h, c)
    constexpr int UN = HD / 4;                       // 16-byte units of a row
    constexpr int NL = F32_BLK * UN / F32_THREADS;   // of K (and of V) a thread loads a block
    static_assert(NL >= 1 && F32_BLK * UN % F32_THREADS == 0 && CHUNK_MULTI % (2 * F32_BLK) == 0, "");
    typedef typename VecN<VC>::T vvec;
    typedef __attribute__((address_space(3))) void lds_t;
    // Two stages, an object each: the compiler then knows that reads of one don't wait for loads
    // into the other.
    __shared__ __attribute__((aligned(16))) F32Stage<HD> st0;
    __shared__ __attribute__((aligned(16))) F32Stage<HD> st1;

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t n = lane & 15u, g = lane >> 4;
    const uint32_t per = TREE ? 1u : F32_WAVES;  // tiles of the workgroup
    const uint32_t kvh = blockIdx.x % p.nkv, nwg = (p.nrb + per - 1) / per;
    const uint32_t wi = nwg - 1u - blockIdx.x / p.nkv;  // latest rows (longest lists) first
    const uint32_t rbi = wave < per ? per * wi + wave : p.nrb, r0 = rbi * p.rb, hd = p.hd, kvd = p.nkv * hd;
    const float* kcb = p.kc + (size_t)kvh * hd;
    const float* vcb = p.vc + (size_t)kvh * hd;
    const uint32_t nrow = n % p.rb, head = n / p.rb;
    const bool valid = head < p.G && r0 + nrow < p.rows;
    uint32_t lo = 0, hi = 0;  // a tree's workgroup: its row's mask
    if (TREE) {
        lo = p.masks[2 * wi];
        hi = p.masks[2 * wi + 1];
    }
    const uint32_t maxlen = TREE ? p.pos + __popc(lo) + __popc(hi) : p.pos + min((wi + 1) * per * p.rb, p.rows);
    const uint32_t len = !valid ? 0u : TREE ? maxlen : p.pos + r0 + nrow + 1u;
    const uint32_t wlen = r0 >= p.rows ? 0u : TREE ? maxlen : p.pos + min(r0 + p.rb, p.rows);  // the wave's longest list

    // This thread's units of a block.
    auto load = [&](F32Stage<HD>& st, uint32_t key0) {
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const uint32_t u0 = F32_THREADS * i + 64 * wave, e = (u0 + lane) / UN, u = (u0 + lane) % UN;
            const uint32_t kk = key0 + e, uk = u ^ (e & 7u);
            const uint32_t s = TREE && kk >= p.pos && kk < maxlen ? p.pos + nth_set_bit(lo, hi, kk - p.pos) : kk;
            const bool ok = kk < maxlen && (uint64_t)s < p.slot_limit;
            const float* ks = ok && 4 * uk < hd ? kcb + (size_t)s * kvd + 4 * uk : p.zero;
            const float* vs = ok && 4 * u < hd ? vcb + (size_t)s * kvd + 4 * u : p.zero;
            __builtin_amdgcn_global_load_lds((const void*)ks, (lds_t*)(&st.k[0][0] + u0), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((const void*)vs, (lds_t*)(&st.v[0][0] + u0), 16, 0, 0);
        }
    };
    load(st0, 0);
    if (tid < (uint32_t)UN) st0.v[F32_BLK][tid] = st1.v[F32_BLK][tid] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 qx[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        qx[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (valid && 16 * j + 4 * g < hd)
            qx[j] = *(const f32x4*)&p.q[((size_t)(r0 + nrow) * p.nh + kvh * p.G + head) * hd + 16 * j + 4 * g];
    }
    float m = -INFINITY, l = 0.0f, RM = -INFINITY, RL = 0.0f;
    f32x4 o[NH * VC], R[NH * VC];
#pragma unroll
    for (int k = 0; k < NH * VC; k++) o[k] = R[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    auto block = [&](F32Stage<HD>& st, F32Stage<HD>& next, uint32_t key0) {
        // This stage's loads are in for everyone, and everyone's reads of the other are done (lgkmcnt:
        // nothing else keeps their last use before the barrier, behind which the loads below go out).
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const bool mine = key0 < wlen;
        f32x4 a0;
        if (mine) a0 = st.k[n][g ^ (n & 7u)];  // before the loads below: it would wait for them
        asm volatile("" : "+v"(a0));
        if (key0 + F32_BLK < maxlen) load(next, key0 + F32_BLK);
        if (!mine) return;
        f32x4 s[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            f32x4 a[8] = {};
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const f32x4 kx = t == 0 && j == 0 ? a0 : st.k[16 * t + n][(4 * j + g) ^ (n & 7u)];
#pragma unroll
                for (int k = 0; k < 4; k++) a[4 * (j % 2) + k] = mfma4(kx[k], qx[j][k], a[4 * (j % 2) + k]);
            }
            s[t] = score_tile(a, p.sc, key0 + 16 * t + 4 * g, len);
        }
        const float cr = softmax_block(s, m, l);
        f32x4 acc[NH * VC] = {};
        const uint32_t left = wlen - key0;
        auto pv = [&](auto whole) {
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t e = 16 * t + 4 * g + i, row = whole || e < left ? e : (uint32_t)F32_BLK;
#pragma unroll
                    for (int h = 0; h < NH; h++) {
                        const vvec v = *((const vvec*)&st.v[row][0] + 16 * h + n);
#pragma unroll
                        for (int k = 0; k < VC; k++) acc[VC * h + k] = mfma4(vec_at(v, k), s[t][i], acc[VC * h + k]);
                    }
                }
        };
        // (two copies: the select in every block cost 2%)
        if (left >= (uint32_t)F32_BLK)
            pv(std::true_type{});
        else
            pv(std::false_type{});
#pragma unroll
        for (int k = 0; k < NH * VC; k++)
#pragma unroll
            for (int i = 0; i < 4; i++) o[k][i] = __builtin_fmaf(o[k][i], cr, acc[k][i]);
    };
    for (uint32_t kb0 = 0; kb0 < maxlen; kb0 += CHUNK_MULTI) {
#pragma unroll 1
        for (uint32_t key0 = kb0; key0 < min(kb0 + CHUNK_MULTI, maxlen); key0 += 2 * F32_BLK) {
            block(st0, st1, key0);
            if (key0 + F32_BLK < maxlen) block(st1, st0, key0 + F32_BLK);
        }
        // The chunk's state folded into the running one (merge_coef, R = R a + c b).
        float fa, fb, mn;
        merge_coef(RM, m, fa, fb, mn);
        RL = RL * fa + slot_sum(l) * fb;
        RM = mn;
#pragma unroll
        for (int k = 0; k < NH * VC; k++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                R[k][i] = R[k][i] * fa + o[k][i] * fb;
                o[k][i] = 0.0f;
            }
        m = -INFINITY;
        l = 0.0f;
    }
    if (!valid) return;
    float* dst = p.out + ((size_t)(r0 + nrow) * p.nh + kvh * p.G + head) * hd;
#pragma unroll
    for (int h = 0; h < NH; h++)
#pragma unroll
        for (int q4 = 0; q4 < VC; q4++) {
            // Lane (n, g): dims 16 VC h + 4 VC g + VC i + k of slot n in o[VC h + k][i].
            const uint32_t d = 16 * VC * h + 4 * VC * g + 4 * q4;
            f32x4 v;
#pragma unroll
            for (int x = 0; x < 4; x++) v[x] = R[VC * h + (4 * q4 + x) % VC][(4 * q4 + x) / VC] / RL;
            if (d < hd) *(f32x4*)(dst + d) = v;
        }
}

static uint32_t ceil_div32(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

constexpr uint64_t F32_SHORT = 128;  // entries (of the farthest list) up to which a call's lists are short

template <int HD, bool SHORT>
static void launch_step(const F32Params& fp, const dim3& grid, const AttnCall& a, hipStream_t s, bool fuse) {
    const dim3 wg(F32_THREADS);
    if (fuse && fp.rows == 1)
        hipExtLaunchKernelGGL((attn_f32_step<HD, 1, SHORT>), grid, wg, 0, s, a.ev_before, a.ev_after, 0, fp);
    else if (fuse)
        hipExtLaunchKernelGGL((attn_f32_step<HD, (int)F32_FUSE_ROWS, SHORT>), grid, wg, 0, s, a.ev_before, a.ev_after, 0, fp);
    else
        hipExtLaunchKernelGGL((attn_f32_step<HD, 0, SHORT>), grid, wg, 0, s, a.ev_before, a.ev_after, 0, fp);
}

template <int HD>
static hipError_t launch_f32(const F32Params& fp, uint32_t blocks, const AttnCall& a, hipStream_t s, bool fuse, bool line,
                             bool is_short) {
    const dim3 grid(blocks), wg(F32_THREADS);
    if (line && fp.tree)
        hipExtLaunchKernelGGL((attn_f32_line<HD, true>), grid, wg, 0, s, a.ev_before, a.ev_after, 0, fp);
    else if (line)
        hipExtLaunchKernelGGL((attn_f32_line<HD, false>), grid, wg, 0, s, a.ev_before, a.ev_after, 0, fp);
    else if (is_short)
        launch_step<HD, true>(fp, grid, a, s, fuse);
    else
        launch_step<HD, false>(fp, grid, a, s, fuse);
    return hipGetLastError();
}

// Tiles from which a line takes the line form: below it the states that a split launch writes
// and the fold reads cost less than CUs left idle or on lists of unequal length (llama-8B heads, 200 rows at
// 300, 400 tiles: 40 us split; 400 rows at 0, 800 tiles: 41 us unsplit).
constexpr uint64_t F32_LINE_TILES = 512;
// Elements of a slot up to which attn_f32_step's 32-bit offsets reach a chunk's slots.
constexpr uint64_t F32_STEP_KVD = 1u << 20;

hipError_t f32_attention(const AttnCall& a, uint64_t kvoff, Workspace& ws, hipStream_t s, const RopeArgs* rope) {
    if (a.rows == 0 || a.nkv == 0 || a.nh % a.nkv != 0 || a.hd == 0 || a.hd % 8 != 0 || a.hd > MAX_HD)
        return hipErrorInvalidValue;
    if (a.tree && a.rows > MAX_ITEMS) return hipErrorInvalidValue;
    if (rope && (a.tree || a.rows > F32_FUSE_ROWS || kvoff != 0 || rope->rope_dim % 2 || rope->rope_dim > a.hd))
        return hipErrorInvalidValue;
    F32Params fp{};
    if (rope) {
        fp.knew = rope->k;
        fp.vnew = rope->v;
        fp.inv_freq = rope->inv_freq;
        fp.positions = rope->positions;
        fp.rope_dim = rope->rope_dim;
        fp.neox = rope->neox;
        fp.qw = rope->q;
    }
    const uint64_t kvd = (uint64_t)a.nkv * a.hd;
    fp.q = a.q;
    fp.kc = (const float*)a.kc + kvoff * kvd;
    fp.vc = (const float*)a.vc + kvoff * kvd;
    fp.out = a.out;
    fp.masks = a.masks;
    fp.tree = a.tree;
    fp.rows = a.rows;
    fp.nh = a.nh;
    fp.nkv = a.nkv;
    fp.hd = a.hd;
    fp.G = a.nh / a.nkv;
    if (fp.G > (uint32_t)F32_SLOTS) return hipErrorInvalidValue;
    fp.pos = a.pos;
    fp.slot_limit = a.slot_limit > kvoff ? a.slot_limit - kvoff : 0;
    fp.zero = (const float*)ws.zero;
    fp.sc = a.scale * LOG2E;
    fp.rb = a.tree ? 1u : std::max<uint32_t>(1u, (uint32_t)F32_SLOTS / fp.G);
    if (fp.rb > a.rows) fp.rb = a.rows;
    fp.nrb = ceil_div32(a.rows, fp.rb);
    // A tree row's list reaches at most 64 entries past pos (its mask's bits); a line's
    // longest is its last row's.
    const uint64_t far = a.tree ? (uint64_t)a.pos + MAX_ITEMS : (uint64_t)a.pos + a.rows;
    fp.nchunk = ceil_div32(far, CHUNK_MULTI);
    const uint64_t groups = (uint64_t)a.nkv * fp.nrb;
    const bool wide = kvd > F32_STEP_KVD;
    bool line = wide || (!a.tree && !rope && groups >= F32_LINE_TILES);
    if (a.tree && !wide && groups >= F32_LINE_TILES && fp.nchunk > 1 && a.rows > 1) {
        // A tree's rows share no list, so the line form (a row a workgroup, one wave of it at work)
        // is not for them: half the rows at a time bounds the states.
        AttnCall h = a;
        h.rows = a.rows / 2;
        h.ev_after = nullptr;
        hipError_t e = f32_attention(h, kvoff, ws, s);
        if (e != hipSuccess) return e;
        h = a;
        h.rows = a.rows - a.rows / 2;
        h.ev_before = nullptr;
        h.q += (size_t)(a.rows / 2) * a.nh * a.hd;
        h.out += (size_t)(a.rows / 2) * a.nh * a.hd;
        h.masks += 2 * (a.rows / 2);
        return f32_attention(h, kvoff, ws, s);
    }
    fp.split = !line && fp.nchunk > 1;
    const uint32_t hdp = a.hd <= 32 ? 32u : a.hd <= 64 ? 64u : a.hd <= 128 ? 128u : 256u;
    if (fp.split) {
        hipError_t e = ws.reserve((size_t)groups * fp.nchunk * F32_SLOTS, hdp);
        if (e == hipSuccess) {
            fp.part_o = ws.o;
            fp.part_ml = ws.ml;
        } else if (ws.fixed) {
            fp.split = 0;  // a fixed workspace too small for the states: the line form, the same bits
            line = true;
        } else {
            return e;
        }
    }
    if (fp.split && a.tree && fp.G <= F32_SLOTS / 2) {
        // Rows share the tiles of the chunks below pos: else each row's tile of G slots fetches and
        // multiplies its own (33 rows at 500 slots, one head a KV head: 61 us, 45 on the vector unit).
        fp.npc = a.pos / CHUNK_MULTI;
        fp.prb = std::min<uint32_t>((uint32_t)F32_SLOTS / fp.G, a.rows);
        fp.npt = ceil_div32(a.rows, fp.prb);
    }
    const uint64_t blocks = line ? (uint64_t)a.nkv * ceil_div32(fp.nrb, a.tree ? 1 : F32_WAVES) : groups * (fp.nchunk - fp.npc) + (uint64_t)a.nkv * fp.npc * fp.npt;
    if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
    hipError_t e;
    if (line && rope) {  // the line form is not fused
        e = rope_append_launch(rope->q, rope->k, rope->v, (void*)a.kc, (void*)a.vc, 0, rope->inv_freq, rope->positions,
                               a.rows, a.nh, a.nkv, a.hd, rope->rope_dim, rope->neox, a.pos, s);
        if (e != hipSuccess) return e;
        rope = nullptr;
    }
    switch (hdp) {
        case 32: e = launch_f32<32>(fp, (uint32_t)blocks, a, s, rope != nullptr, line, far <= F32_SHORT); break;
        case 64: e = launch_f32<64>(fp, (uint32_t)blocks, a, s, rope != nullptr, line, far <= F32_SHORT); break;
        case 128: e = launch_f32<128>(fp, (uint32_t)blocks, a, s, rope != nullptr, line, far <= F32_SHORT); break;
        default: e = launch_f32<256>(fp, (uint32_t)blocks, a, s, rope != nullptr, line, far <= F32_SHORT); break;
    }
    if (e != hipSuccess || !fp.split) return e;
    CombineParams cp{};
    cp.long_fold = ws.combine_long;
    cp.zero = ws.zero;
    cp.out = a.out;
    cp.part_o = ws.o;
    cp.part_ml = ws.ml;
    cp.nh = a.nh;
    cp.nkv = a.nkv;
    cp.hd = a.hd;
    cp.G = fp.G;
    cp.slots = F32_SLOTS;
    cp.slots_out = F32_SLOTS;
    cp.shared = 1;
    cp.rows = a.rows;
    cp.rb = fp.rb;
    cp.nrb = fp.nrb;
    cp.nchunk = fp.nchunk;
    if (rope) {
        cp.fuse = 1;
        cp.qw = rope->q;
        cp.inv_freq = rope->inv_freq;
        cp.positions = rope->positions;
        cp.rope_dim = rope->rope_dim;
        cp.neox = rope->neox;
    }
    return combine_launch(cp, (uint32_t)groups, a.hd, s);
}

}  // namespace bchip
