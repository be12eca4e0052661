// The rest of bc-infer's layer on the GPU: the GGUF block-format matrix product
// (crates/bc-infer/src/gpu/kernels.h:51-214, entry cuda.cu:77-79), RMSNorm (kernels.h:216-225,
// cuda.cu:80) and the elementwise ops (kernels.h:327-330, cuda.cu:86-88).
//
// Five kernels share the product: k_matmul_row (one input row of the block formats), k_matmul_mm
// (batches), k_matmul_units (small batches off a multiple of 256 columns) and k_matmul_tile (large
// batches) on the matrix cores, the last three in one arithmetic; k_matmul (plain types, and one row
// that k_matmul_row does not take) on the vector unit. Weights stay in their ggml blocks, rows of
// whole blocks (row_bytes = cols / block_weights * block_bytes).
//
// k_matmul: every format is read a "group" of 32 weights at a time. A wave owns R weight rows and its 64 lanes take the row's groups, one each per
// column tile: per group the lane loads its rows' packed bytes and its input values (up to
// NB input rows), unpacks each row's 32 quants and sums in a fixed order. The 64 lane sums meet in a
// fixed butterfly. In each kernel an input row's result depends on that row alone, never on how
// many rows share the batch, and reruns give the same bits (the reference kernel's properties,
// kernels.h:9-11).
#include "common.hpp"
#include "internal.hpp"

#include <algorithm>
#include <type_traits>

namespace bchip {

// ggml type numbers (quant.rs:35-49).
enum : uint32_t {
    G_F32 = 0, G_F16 = 1, G_Q4_0 = 2, G_Q4_1 = 3, G_Q5_0 = 6, G_Q5_1 = 7, G_Q8_0 = 8,
    G_Q4K = 12, G_Q5K = 13, G_Q6K = 14, G_BF16 = 30,
};

bool ggml_block(uint32_t ty, uint32_t& weights, uint32_t& bytes) {
    switch (ty) {
        case G_F32: weights = 1; bytes = 4; return true;
        case G_F16: case G_BF16: weights = 1; bytes = 2; return true;
        case G_Q4_0: weights = 32; bytes = 18; return true;
        case G_Q4_1: weights = 32; bytes = 20; return true;
        case G_Q5_0: weights = 32; bytes = 22; return true;
        case G_Q5_1: weights = 32; bytes = 24; return true;
        case G_Q8_0: weights = 32; bytes = 34; return true;
        case G_Q4K: weights = 256; bytes = 144; return true;
        case G_Q5K: weights = 256; bytes = 176; return true;
        case G_Q6K: weights = 256; bytes = 210; return true;
        default: return false;
    }
}

constexpr int NB = 8;  // input rows a pass (grid.y) takes

__device__ __forceinline__ float h2f(uint32_t bits16) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16);
}
__device__ __forceinline__ uint32_t ld16(const uint8_t* p) { return *(const uint16_t*)p; }
// Four bytes at a 2-byte-aligned address.
__device__ __forceinline__ uint32_t ld32h(const uint8_t* p) { return ld16(p) | (ld16(p + 2) << 16); }
__device__ __forceinline__ uint32_t ld32(const uint8_t* p) { return *(const uint32_t*)p; }
__device__ __forceinline__ float i8f(uint32_t b) { return (float)(int8_t)(uint8_t)b; }

// A group's bytes are loaded first (packed, PK<TY> dwords: a few registers a group, so a
// wave can hold several rows' groups in flight) and unpacked just before use.
template <uint32_t TY>
constexpr int PK = TY == G_F32 ? 32 : (TY == G_F16 || TY == G_BF16) ? 16 : (TY == G_Q4_0 || TY == G_Q4_1) ? 5
                 : (TY == G_Q5_0 || TY == G_Q5_1) ? 6 : TY == G_Q8_0 ? 9 : TY == G_Q4K ? 12 : TY == G_Q5K ? 20 : 17;

template <uint32_t TY>
__device__ __forceinline__ void group_load(const uint8_t* __restrict__ row, uint32_t g, uint32_t (&pk)[PK<TY>]) {
    if constexpr (TY == G_F32 || TY == G_F16 || TY == G_BF16) {
        const uint4* p = (const uint4*)(row + (size_t)g * (TY == G_F32 ? 128 : 64));
#pragma unroll
        for (int k = 0; k < PK<TY> / 4; k++) {
            const uint4 v = p[k];
            pk[4 * k] = v.x; pk[4 * k + 1] = v.y; pk[4 * k + 2] = v.z; pk[4 * k + 3] = v.w;
        }
    } else if constexpr (TY == G_Q8_0) {
        const uint8_t* b8 = row + (size_t)g * 34;
        pk[0] = ld16(b8);
#pragma unroll
        for (int k = 0; k < 8; k++) pk[1 + k] = ld32h(b8 + 2 + 4 * k);
    } else if constexpr (TY == G_Q4_0 || TY == G_Q5_0 || TY == G_Q4_1 || TY == G_Q5_1) {
        constexpr bool Q41 = TY == G_Q4_1 || TY == G_Q5_1, FIVE = TY == G_Q5_0 || TY == G_Q5_1;
        constexpr uint32_t BS = TY == G_Q4_0 ? 18 : TY == G_Q4_1 ? 20 : TY == G_Q5_0 ? 22 : 24;
        const uint8_t* bb = row + (size_t)g * BS;
        pk[0] = Q41 ? ld32(bb) : ld16(bb);  // d (and m)
        if constexpr (FIVE) pk[5] = ld32h(bb + (Q41 ? 4 : 2));
        const uint8_t* qs = bb + (Q41 ? 4 : 2) + (FIVE ? 4 : 0);
#pragma unroll
        for (int k = 0; k < 4; k++) pk[1 + k] = Q41 ? ld32(qs + 4 * k) : ld32h(qs + 4 * k);
    } else if constexpr (TY == G_Q4K || TY == G_Q5K) {
        const uint8_t* bb = row + (size_t)(g / 8) * (TY == G_Q4K ? 144 : 176);
        const uint32_t c = (g % 8) / 2;
#pragma unroll
        for (int k = 0; k < 4; k++) pk[k] = ld32(bb + 4 * k);  // d, dmin, the 12 scale bytes
        const uint8_t* qs = bb + (TY == G_Q4K ? 16 : 48) + 32 * c;
#pragma unroll
        for (int k = 0; k < 8; k++) pk[4 + k] = ld32(qs + 4 * k);
        if constexpr (TY == G_Q5K) {
#pragma unroll
            for (int k = 0; k < 8; k++) pk[12 + k] = ld32(bb + 16 + 4 * k);
        }
    } else {  // Q6K
        const uint8_t* bb = row + (size_t)(g / 8) * 210;
        const uint32_t sub = g % 8, hh = sub / 4, qr = sub % 4;
        const uint8_t* ql = bb + 64 * hh + ((qr & 1u) ? 32 : 0);
        const uint8_t* qh = bb + 128 + 32 * hh;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            pk[k] = ld32h(ql + 4 * k);
            pk[8 + k] = ld32h(qh + 4 * k);
        }
        pk[16] = ld16(bb + 192 + 8 * hh + 2 * qr) | (ld16(bb + 208) << 16);
    }
}

// Group g's quants and per-half affine maps from its packed bytes: weight j = a[h] * q[j] +
// b[h] for h = j / 16 (quant.rs:150-259's values: Q4_0 (q - 8) d, Q4_1 q d + m, Q5_0
// (q - 16) d, Q5_1 q d + m, Q8_0 q d, Q4K/Q5K ds q - dm, Q6K d_h (q - 32); the plain types
// are their values with a = 1, b = 0). The product then needs per half only sum(q x) and
// sum(x): one conversion and one FMA a weight, not a dequantization and a product.
template <uint32_t TY>
constexpr bool plain_type() {
    return TY == G_F32 || TY == G_F16 || TY == G_BF16;
}

// Bytes 0..3 of v as floats (the hardware's byte-to-float conversions).
__device__ __forceinline__ void bytes4(uint32_t v, float* q) {
    q[0] = (float)(v & 255u);
    q[1] = (float)((v >> 8) & 255u);
    q[2] = (float)((v >> 16) & 255u);
    q[3] = (float)(v >> 24);
}

template <uint32_t TY>
__device__ __forceinline__ void group_unpack(const uint32_t (&pk)[PK<TY>], uint32_t g, float (&q)[32], float (&a)[2],
                                             float (&b)[2]) {
    if constexpr (TY == G_F32) {
#pragma unroll
        for (int j = 0; j < 32; j++) q[j] = __uint_as_float(pk[j]);
    } else if constexpr (TY == G_F16 || TY == G_BF16) {
#pragma unroll
        for (int j = 0; j < 16; j++) {
            if constexpr (TY == G_F16) {
                q[2 * j] = h2f(pk[j] & 0xffffu);
                q[2 * j + 1] = h2f(pk[j] >> 16);
            } else {
                q[2 * j] = __uint_as_float(pk[j] << 16);
                q[2 * j + 1] = __uint_as_float(pk[j] & 0xffff0000u);
            }
        }
    } else if constexpr (TY == G_Q8_0) {
#pragma unroll
        for (int k = 0; k < 8; k++)
#pragma unroll
            for (int j = 0; j < 4; j++) q[4 * k + j] = i8f(pk[1 + k] >> (8 * j));
        a[0] = a[1] = h2f(pk[0]);
        b[0] = b[1] = 0.0f;
    } else if constexpr (TY == G_Q4_0 || TY == G_Q5_0 || TY == G_Q4_1 || TY == G_Q5_1) {
        // element j in byte j's low nibble, j + 16 in its high nibble; Q5 adds bit j of qh as
        // bit 4 of element j
        constexpr bool Q41 = TY == G_Q4_1 || TY == G_Q5_1, FIVE = TY == G_Q5_0 || TY == G_Q5_1;
        const float d = h2f(pk[0] & 0xffffu);
        const float m = Q41 ? h2f(pk[0] >> 16) : 0.0f;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            uint32_t lo = pk[1 + k] & 0x0f0f0f0fu, hi = (pk[1 + k] >> 4) & 0x0f0f0f0fu;
            if constexpr (FIVE) {
                // bits 4k .. 4k+3 of qh to bit 4 of bytes 0..3; bits 16 + 4k .. likewise
                const uint32_t qh = pk[5];
                const uint32_t l4 = (qh >> (4 * k)) & 15u, h4 = (qh >> (16 + 4 * k)) & 15u;
                lo |= ((l4 & 1u) << 4) | ((l4 & 2u) << 11) | ((l4 & 4u) << 18) | ((l4 & 8u) << 25);
                hi |= ((h4 & 1u) << 4) | ((h4 & 2u) << 11) | ((h4 & 4u) << 18) | ((h4 & 8u) << 25);
            }
            bytes4(lo, &q[4 * k]);
            bytes4(hi, &q[16 + 4 * k]);
        }
        a[0] = a[1] = d;
        b[0] = b[1] = Q41 ? m : (TY == G_Q4_0 ? -8.0f : -16.0f) * d;
    } else if constexpr (TY == G_Q4K || TY == G_Q5K) {
        // 256 weights a block in 4 chunks of 64: group 2c is chunk c's low nibbles, 2c + 1 its
        // high nibbles (Q5K: plus bit 2c + hi of each qh byte, as bit 4).
        const uint32_t sub = g % 8, c = sub / 2, hi = sub % 2;
        const float d = h2f(pk[0] & 0xffffu), dmin = h2f(pk[0] >> 16);
        auto sbyte = [&](uint32_t k) { return (pk[1 + k / 4] >> (8 * (k % 4))) & 255u; };  // scales[k]
        float sc, mn;
        if (sub < 4) {  // quant.rs:136-146
            sc = (float)(sbyte(sub) & 63u);
            mn = (float)(sbyte(sub + 4) & 63u);
        } else {
            sc = (float)((sbyte(sub + 4) & 15u) | ((sbyte(sub - 4) >> 6) << 4));
            mn = (float)((sbyte(sub + 4) >> 4) | ((sbyte(sub) >> 6) << 4));
        }
#pragma unroll
        for (int k = 0; k < 8; k++) {
            uint32_t v = (pk[4 + k] >> (4 * hi)) & 0x0f0f0f0fu;
            if constexpr (TY == G_Q5K) v |= ((pk[12 + k] >> (2 * c + hi)) & 0x01010101u) << 4;
            bytes4(v, &q[4 * k]);
        }
        a[0] = a[1] = d * sc;
        b[0] = b[1] = -(dmin * mn);
    } else {  // Q6K: ql nibble qr / 2, qh bits 2qr, scales for weights 0..15 and 16..31
        const uint32_t qr = (g % 8) % 4, shift = qr < 2 ? 0 : 4;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t v = ((pk[k] >> shift) & 0x0f0f0f0fu) | (((pk[8 + k] >> (2 * qr)) & 0x03030303u) << 4);
            bytes4(v, &q[4 * k]);
        }
        const float d = h2f(pk[16] >> 16);
        a[0] = d * i8f(pk[16] & 255u);
        a[1] = d * i8f((pk[16] >> 8) & 255u);
        b[0] = -32.0f * a[0];
        b[1] = -32.0f * a[1];
    }
}

// Sum over a wave of one value per lane, the same butterfly for every call.
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    return v;
}

struct MatmulParams {
    const uint8_t* w;
    const float* x;
    float* out;
    uint32_t rows, cols, n, row_bytes;
};

// out[i][r] = sum_c W[r][c] x[i][c]: workgroup (blockIdx.x) = MM_WAVES waves x R weight rows,
// blockIdx.y = input rows i0 .. i0 + NBT. The input rows pass through LDS in column tiles of
// 64 groups (one group a lane), read from HBM once per workgroup with coalesced loads and
// stored with a padded group stride (XS floats) so that each lane's 16-byte reads of its
// group fall on distinct banks; each lane's packed weights for the tile are loaded before
// the tile, so the two latencies overlap. Per lane, group and input row: the two half sums
// of q x (FMA chains, weights in order) and of x, then acc += a0 sq0 + a1 sq1 + b0 sx0 +
// b1 sx1 (in that order, as FMAs); the 64 lane sums meet in a fixed butterfly. R only sets
// which rows a wave holds, not a row's arithmetic.
constexpr int XS = 36;           // LDS floats per group of 32 inputs
constexpr int TILE_GROUPS = 64;  // groups per column tile: one per lane
constexpr int MM_WAVES = 4;      // waves a workgroup

template <uint32_t TY, int NBT, int R>
__global__ __launch_bounds__(64 * MM_WAVES) void k_matmul(const MatmulParams p) {
    // nb tiles of TILE_GROUPS * XS floats (dynamic: a one-row pass takes 9 KB, so more
    // workgroups share a CU).
    extern __shared__ __attribute__((aligned(16))) float xs_dyn[];
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r0 = (blockIdx.x * MM_WAVES + wave) * R;
    const uint32_t i0 = blockIdx.y * NBT;
    const uint32_t nb = min((uint32_t)NBT, p.n - i0);
    const uint32_t groups = p.cols / 32;
    float acc[NBT][R];
#pragma unroll
    for (int i = 0; i < NBT; i++)
#pragma unroll
        for (int r = 0; r < R; r++) acc[i][r] = 0.0f;
    // Rows past the matrix read its last row (their sums are never stored).
    const uint8_t* rowp[R];
#pragma unroll
    for (int r = 0; r < R; r++) rowp[r] = p.w + (size_t)min(r0 + r, p.rows - 1) * p.row_bytes;
    for (uint32_t t0 = 0; t0 < groups; t0 += TILE_GROUPS) {
        const uint32_t tg = min((uint32_t)TILE_GROUPS, groups - t0);
        // This lane's weights first, packed (lanes past the tile read its first group); then
        // the tile of every input row: float4 e of it is group e / 8, quarter e % 8.
        const uint32_t g = t0 + (lane < tg ? lane : 0u);
        uint32_t pk[R][PK<TY>];
#pragma unroll
        for (int r = 0; r < R; r++) group_load<TY>(rowp[r], g, pk[r]);
        __syncthreads();
        for (uint32_t e = threadIdx.x; e < nb * tg * 8; e += 64 * MM_WAVES) {
            const uint32_t i = e / (tg * 8), f = e % (tg * 8);
            const float4 v = *(const float4*)(p.x + (size_t)(i0 + i) * p.cols + 32 * t0 + 4 * f);
            *(float4*)&xs_dyn[i * TILE_GROUPS * XS + (f / 8) * XS + 4 * (f % 8)] = v;
        }
        __syncthreads();
        if (lane >= tg) continue;
        // One row's group against one input row's values (the same FMA order in both loop
        // nests below, so a row gets the same bits either way).
        auto dot = [&](const float (&q)[32], const float (&a)[2], const float (&b)[2], const float (&xv)[32],
                       float sx0, float sx1, float& acc_ir) {
            if constexpr (plain_type<TY>()) {
                float sum = acc_ir;
#pragma unroll
                for (int j = 0; j < 32; j++) sum = __builtin_fmaf(q[j], xv[j], sum);
                acc_ir = sum;
            } else {
                float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
                for (int j = 0; j < 16; j++) {
                    s0 = __builtin_fmaf(q[j], xv[j], s0);
                    s1 = __builtin_fmaf(q[16 + j], xv[16 + j], s1);
                }
                float t = __builtin_fmaf(a[0], s0, acc_ir);
                t = __builtin_fmaf(a[1], s1, t);
                t = __builtin_fmaf(b[0], sx0, t);
                acc_ir = __builtin_fmaf(b[1], sx1, t);
            }
        };
        auto read_x = [&](int i, float (&xv)[32], float& sx0, float& sx1) {
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float4 v = *(const float4*)&xs_dyn[i * TILE_GROUPS * XS + lane * XS + 4 * k];
                xv[4 * k] = v.x; xv[4 * k + 1] = v.y; xv[4 * k + 2] = v.z; xv[4 * k + 3] = v.w;
            }
            sx0 = sx1 = 0.0f;
            if constexpr (!plain_type<TY>()) {
#pragma unroll
                for (int j = 0; j < 16; j++) {
                    sx0 += xv[j];
                    sx1 += xv[16 + j];
                }
            }
        };
        if constexpr (NBT == 1) {
            // One input row: its values once, each row unpacked in turn.
            float xv[32], sx0, sx1;
            read_x(0, xv, sx0, sx1);
#pragma unroll
            for (int r = 0; r < R; r++) {
                float q[32], a[2], b[2];
                group_unpack<TY>(pk[r], g, q, a, b);
                dot(q, a, b, xv, sx0, sx1, acc[0][r]);
            }
        } else {
            // A batch: each row unpacked once, the input rows' values read again from LDS.
            float sx[NBT][2];
#pragma unroll
            for (int i = 0; i < NBT; i++) {
                if (i < (int)nb) {
                    float xv[32];
                    read_x(i, xv, sx[i][0], sx[i][1]);
                }
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                float q[32], a[2], b[2];
                group_unpack<TY>(pk[r], g, q, a, b);
#pragma unroll
                for (int i = 0; i < NBT; i++) {
                    if (i < (int)nb) {
                        float xv[32], u0, u1;
                        read_x(i, xv, u0, u1);
                        dot(q, a, b, xv, sx[i][0], sx[i][1], acc[i][r]);
                    }
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < NBT; i++) {
        if (i < (int)nb) {
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float s = wave_sum(acc[i][r]);
                if (lane == 0 && r0 + r < p.rows) p.out[(size_t)(i0 + i) * p.rows + r0 + r] = s;
            }
        }
    }
}

// ---------------------------------------------------------------------------------------
// Batched product on the matrix cores (n >= MM_MIN input rows; the reference switches its
// batches to a matrix-unit product the same way, gpu/mod.rs:33-41, metal.rs:153-197).
// In the affine form, group g of weight row r is w = a q + b, q a small integer; so
// sum_k w x = a sum q x + b sum x. The MFMAs compute sum q x with x split into two f16 parts:
// a unit of 256 columns of an input row is scaled by a power of two s that puts its largest
// |x| in [2^14, 2^15), hi = f16(x s), lo = f16((x s - hi) 2^12): 22 bits of every x within 2^-29
// of the unit's largest and an absolute error below 2^-51 of it for the rest (with lo unscaled
// 2^-17 and 2^-39: columns 1e6 below others that met weights of 0 were 4e-7 off, so 1.1e-7), each
// product exact in f32, f32-level sums. A unit's hi and lo sums meet at its end, the lo sum
// times 2^-12. (Q6K, whose MFMAs add both, keeps lo unscaled: weights times 2^-12 over lo cost
// its tile kernel 4%, and its vector-unit pass lost more in such columns, 4e-3.)
//
// k_matmul_mm: a workgroup is W waves of 16 weight rows, eight input rows and a K range of
// at most MM_K units. The range's x is staged once in LDS as 16 A rows: rows 0 .. 7 the eight
// inputs' hi, rows 8 .. 15 their lo, so one v_mfma_f32_16x16x32_f16 over group g gives D[i][l]
// = sum hi_i q (i < 8) and sum lo_{i-8} q (i >= 8), each in a chain of its own, for the
// wave's 16 rows at once. Lane 16 c + l holds 8 weights of group g of row r0 + l (8c .. 8c +
// 7) as its B operand, unpacked from the ggml bytes in registers, in the order 0, 2,
// 1, 3, 4, 6, 5, 7 (pairs of bytes 0, 2 and 1, 3 of a dword make the f16 pairs directly;
// staged x is permuted alike, and the MFMA's sum over k is the group's either way): each
// field is put under the f16 exponent of 1024 (one v_and_or_b32 for a pair of nibbles,
// v_perm_b32 for a pair of bytes) and one packed f16 subtraction takes 1024 and the format's
// fixed offset away (Q4_0 8, Q5_0 16, Q6K 32, Q8_0 -128 after a sign flip). Q6K has a scale
// a 16 weights: its two MFMAs a group take one half each, lane c holding weights 4c .. 4c + 3
// of the half twice, over x's hi and over its lo (A rows 8 .. 15 are inputs 0 .. 7 again). D[4c + i][l] is in lane 16 c + l.
// Accumulation, per output element, in this order whatever kernel computes it:
//   T_hi, T_lo = the MFMAs of a group over hi and over lo (Q4K, Q5K, F16: chained over the
//   unit's groups; Q6K: one T of a half, hi and lo in one MFMA)
//   t_hi += a T_hi, t_lo += a T_lo per group, zeroed each unit (Q4K, Q5K, F16: t = T)
//   t = t_hi + 2^-12 t_lo, one FMA (Q6K: t += a T per half)
//   t = d t (Q4K, Q5K), then t += the unit's b sum x terms; p += t / s per unit
//   out = the K splits' p added in split order.
// The b sum x terms (Q4_1, Q5_1: m; Q4K, Q5K: -dmin m_j) are one more MFMA a unit: A = the
// eight groups' sums of (hi + lo) / 32 in three f16 parts (33 bits), B = the m's three times over
// (Q4K, Q5K: the last two parts times 2^12 over m 2^-12, a floor of 2^-52 of the unit's largest
// |x|, else 2^-40: small groups beside columns 1e6 larger, 2.5e-6 off without).
// The units' bytes are loaded MM_PF units ahead. K splits: their number depends on rows and
// cols only; one workgroup runs the splits one after another or ks workgroups run them at
// once and the last to finish (a device counter per tile) adds them: an input row's bits
// depend on that row alone, never on n or its place in the batch.
constexpr uint32_t MM_MIN = 2;     // batches of at least this many rows take the matrix cores (MM_FROM)
// Units (256 columns) a K split at most: the staged x takes 16 rows x (256 MM_K + 8) halves of
// LDS (rows 8 banks apart measured 0.6 us a call better than 4); the K-quants also pass each unit's
// bytes through LDS, so their splits are shorter.
template <uint32_t TY>
constexpr bool MM_LDSP = TY != G_F16;  // units pass through LDS (all block formats)
template <uint32_t TY>
constexpr uint32_t MM_K = MM_LDSP<TY> ? 4 : 8;
template <uint32_t TY>
constexpr uint32_t MM_XS = MM_K<TY> * 256 + 16;
constexpr uint32_t MM_PAR = MATMUL_COUNTERS;  // tiles (W x 16 rows x 8 inputs) up to which K splits run in parallel

template <uint32_t TY>
constexpr bool mm_type() {
    return TY == G_F16 || TY == G_Q8_0 || TY == G_Q4_0 || TY == G_Q4_1 || TY == G_Q5_0 || TY == G_Q5_1 ||
           TY == G_Q4K || TY == G_Q5K || TY == G_Q6K;
}
// x's order: 0 as it is (F16), 1 in pairs (0, 2, 1, 3 of each four), 2 the same
// with hi and lo of each four columns together (Q6K).
template <uint32_t TY>
constexpr int tl_order() {
    return TY == G_F16 ? 0 : TY == G_Q6K ? 2 : 1;
}
// Formats with b sum x terms.
template <uint32_t TY>
constexpr bool mm_sum() {
    return TY == G_Q4_1 || TY == G_Q5_1 || TY == G_Q4K || TY == G_Q5K;
}
// Dwords a lane loads of one unit (8 groups) of its row, and holds of it after mm_fix.
template <uint32_t TY>
constexpr int MW = TY == G_F16 ? 32 : TY == G_Q8_0 ? 20 : TY == G_Q6K ? 16 : 12;
template <uint32_t TY>
constexpr int MWD = TY == G_Q5K ? 14 : TY == G_Q6K ? 29 : MW<TY>;
// Units loaded ahead; waves a workgroup (eight where the registers allow four waves a SIMD).
template <uint32_t TY>
constexpr int MM_PF = 2;
template <uint32_t TY>
constexpr int MM_W = MM_LDSP<TY> ? 8 : 4;
// Bytes of a unit.
template <uint32_t TY>
constexpr uint32_t MM_UB = TY == G_F16 ? 512 : TY == G_Q8_0 ? 272 : TY == G_Q4_0 ? 144 : TY == G_Q4_1 ? 160
                         : TY == G_Q5_0 ? 176 : TY == G_Q5_1 ? 192 : TY == G_Q4K ? 144 : TY == G_Q5K ? 176 : 210;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// The lane order of a dword's four bytes: 0, 2, 1, 3.
// Bytes of v as f16 values 1024 + b - off, in that order (two f16 pairs).
__device__ __forceinline__ u32x2 bytes_f16(uint32_t v, half2 off) {
    const uint32_t e0 = __builtin_amdgcn_perm(0x64646464u, v, 0x04020400u);  // (0x6400 | b0, 0x6400 | b2)
    const uint32_t e1 = __builtin_amdgcn_perm(0x64646464u, v, 0x04030401u);  // (0x6400 | b1, 0x6400 | b3)
    const half2 h0 = __builtin_bit_cast(half2, e0) - off, h1 = __builtin_bit_cast(half2, e1) - off;
    return u32x2{__builtin_bit_cast(uint32_t, h0), __builtin_bit_cast(uint32_t, h1)};
}
__device__ __forceinline__ half8 bytes8_f16(uint32_t v0, uint32_t v1, half2 off) {
    const u32x2 a = bytes_f16(v0, off), b = bytes_f16(v1, off);
    return __builtin_bit_cast(half8, u32x4{a[0], a[1], b[0], b[1]});
}
// The field under m (within each 16 bits: 0x000f000f, 0x00f000f0) of bytes 0, 2 of v as f16
// 1024 + f - off (exact): the field under the exponent of 1024 (one v_and_or_b32), then one
// packed subtraction. (Fields as f16 subnormals, f 2^-24, would need no subtraction, but the
// matrix cores multiply subnormals less exactly: about 1.7e-6 of a row's scale against 2e-7.)
// (v & m) | e in one v_and_or_b32 (m in a VGPR, e an SGPR: the instruction may read one
// SGPR and no literal, so the compiler otherwise splits it in two).
__device__ __forceinline__ uint32_t and_or(uint32_t v, uint32_t m, uint32_t e) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "v"(m), "s"(e));
    return r;
}
__device__ __forceinline__ uint32_t field_pair(uint32_t v, uint32_t m, half2 off, uint32_t extra = 0u) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2, and_or(v, m, extra | 0x64006400u)) - off);
}
// As field_pair, times a scale in one packed FMA: (1024 + f) c1 + c2 with c2 = -1024 c1, exact
// while f c1 is an f16 integer (K-quant sub-block scale times field: at most 63 x 31).
__device__ __forceinline__ uint32_t field_pair_sc(uint32_t v, uint32_t m, half2 c1, half2 c2, uint32_t extra = 0u) {
    const half2 e = __builtin_bit_cast(half2, and_or(v, m, extra | 0x64006400u));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(e, c1, c2));
}
// Bytes 0, 2, then 1, 3 of two dwords.
__device__ __forceinline__ half8 fields8(uint32_t v0, uint32_t v1, uint32_t m, half2 off) {
    return __builtin_bit_cast(half8, u32x4{field_pair(v0, m, off), field_pair(v0 >> 8, m, off),
                                           field_pair(v1, m, off), field_pair(v1 >> 8, m, off)});
}
// Four bits to bit 4 of bytes 0..3.
__device__ __forceinline__ uint32_t bit4_spread(uint32_t b4) { return ((b4 * 0x00204081u) & 0x01010101u) << 4; }
// Lane (c, row) loads of unit u (8 groups) of its row.
template <uint32_t TY>
__device__ __forceinline__ void mm_load(const uint8_t* __restrict__ row, uint32_t u, uint32_t c,
                                        uint32_t (&d)[MW<TY>]) {
    if constexpr (TY == G_F16) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const u32x4 v = *(const u32x4*)(row + (size_t)(8 * u + j) * 64 + 16 * c);
            d[4 * j] = v[0]; d[4 * j + 1] = v[1]; d[4 * j + 2] = v[2]; d[4 * j + 3] = v[3];
        }
    } else if constexpr (TY == G_Q8_0) {
        // Row-contiguous lane order as the K-quants' (below): 17 pieces a unit, lane quad q
        // takes pieces 4 l + (lane & 3), l < 5 (the repeats past the unit are its last piece).
        const uint8_t* bb = row + (size_t)u * 272;
        const uint32_t pq = threadIdx.x & 3u;
#pragma unroll
        for (int l = 0; l < 5; l++) {
            const u32x4 v = *(const u32x4*)(bb + 16 * min(4 * l + pq, 16u));
            d[4 * l] = v[0]; d[4 * l + 1] = v[1]; d[4 * l + 2] = v[2]; d[4 * l + 3] = v[3];
        }
    } else if constexpr (TY == G_Q4_0 || TY == G_Q4_1 || TY == G_Q5_0 || TY == G_Q5_1) {
        // row-contiguous lane order, as the K-quants' below (9 to 12 pieces a unit)
        constexpr uint32_t NP = MM_UB<TY> / 16;
        const uint8_t* bb = row + (size_t)u * MM_UB<TY>;
        const uint32_t pq = threadIdx.x & 3u;
#pragma unroll
        for (int l = 0; l < 3; l++) {
            const u32x4 v = *(const u32x4*)(bb + 16 * min(4 * l + pq, NP - 1));
            d[4 * l] = v[0]; d[4 * l + 1] = v[1]; d[4 * l + 2] = v[2]; d[4 * l + 3] = v[3];
        }
    } else if constexpr (TY == G_Q4K || TY == G_Q5K) {
        // Row-contiguous lane order (the memory path coalesces consecutive lanes: 64 bytes of
        // one row a lane quad), 16-byte pieces 4 l + (lane & 3) of the unit for l < 3 (the last
        // load's pieces past the unit repeat its last); `row` is the lane quad's row, and
        // mm_fix moves the pieces through LDS into the matrix-core layout.
        constexpr uint32_t NP = MM_UB<TY> / 16;  // pieces a unit: 9 (Q4K), 11 (Q5K)
        const uint8_t* bb = row + (size_t)u * MM_UB<TY>;
        const uint32_t pq = threadIdx.x & 3u;
#pragma unroll
        for (int l = 0; l < 3; l++) {
            const u32x4 v = *(const u32x4*)(bb + 16 * min(4 * l + pq, NP - 1));
            d[4 * l] = v[0]; d[4 * l + 1] = v[1]; d[4 * l + 2] = v[2]; d[4 * l + 3] = v[3];
        }
    } else {  // Q6K, row-contiguous lane order: the 16-byte pieces from the unit's start
        // rounded down to 16 (at most 14 pieces hold its 210 bytes; a lane quad takes pieces
        // 4 l + (lane & 3), l < 4, those past the last that holds unit bytes repeat it, so no
        // read leaves the 16-byte blocks the unit touches)
        const uint8_t* bb = row + (size_t)u * 210;
        const uintptr_t a0 = (uintptr_t)bb & ~(uintptr_t)15;
        const uint32_t km = (uint32_t)((uintptr_t)bb + 209 - a0) / 16, pq = threadIdx.x & 3u;
#pragma unroll
        for (int l = 0; l < 4; l++) {
            const u32x4 v = *(const u32x4*)(a0 + 16 * min(4 * l + pq, km));
            d[4 * l] = v[0]; d[4 * l + 1] = v[1]; d[4 * l + 2] = v[2]; d[4 * l + 3] = v[3];
        }
    }
}

// After a unit's loads land (K-quants): each lane quad's three pieces go to the wave's LDS
// rows (row q = lane / 4, the unit's 16-byte pieces, piece p at slot p ^ ((q >> 2) & 3) of a
// 192-byte row: the quads' 64-byte writes and the 16 rows' reads of one piece fall on
// distinct banks), and each lane reads back what the matrix-core layout gives it: the header
// (d, dmin, scales) and slice c of each 32-byte qs chunk (Q5K also qh bytes 8c .. 8c + 7),
// into d[0..3], d[4 + 2k..5 + 2k] (chunk k) and d[12..13].
// LDS bytes a row of a unit: K-quants 192 (swizzled pieces), Q8_0 272 (the unit as it is:
// a stride of 68 dwords puts the 16 rows' dword reads of one offset on distinct banks).
// The 32-weight formats' units keep their bytes as they are, in rows of an odd number of
// 16-byte pieces (Q4_1, Q5_1 padded by one) for the same bank spread.
template <uint32_t TY>
constexpr uint32_t MM_WT = TY == G_Q8_0 ? 272 : TY == G_Q6K ? 240 : TY == G_Q4_0 ? 144 : TY == G_Q4_1 ? 176
                         : TY == G_Q5_0 ? 176 : TY == G_Q5_1 ? 208 : 192;
// s: the lane's loads; d: what mm_unit and mm_group read; sq, sm: the lane quad's and the
// lane's own row's unit start modulo 16 (Q6K).
template <uint32_t TY>
__device__ __forceinline__ void mm_fix(const uint32_t (&s)[MW<TY>], uint32_t (&d)[MWD<TY>], uint8_t* wt, uint32_t c,
                                       uint32_t rl, uint32_t sq, uint32_t sm) {
    if constexpr (!MM_LDSP<TY>) {
#pragma unroll
        for (int k = 0; k < MW<TY>; k++) d[k] = s[k];
    }
    if constexpr (TY == G_Q8_0 || TY == G_Q4_0 || TY == G_Q4_1 || TY == G_Q5_0 || TY == G_Q5_1) {
        // the unit to the LDS rows as it is; mm_group reads each group from there
        constexpr uint32_t NP = MM_UB<TY> / 16;
        const uint32_t q = (threadIdx.x & 63u) >> 2, pq = threadIdx.x & 3u;
#pragma unroll
        for (int l = 0; l < MW<TY> / 4; l++)
            if (4 * l + pq < NP)
                *(u32x4*)(wt + q * MM_WT<TY> + 16 * (4 * l + pq)) = u32x4{s[4 * l], s[4 * l + 1], s[4 * l + 2], s[4 * l + 3]};
        if constexpr (TY == G_Q4_1 || TY == G_Q5_1) {  // the unit's eight m's (the b terms)
            constexpr uint32_t BS = TY == G_Q4_1 ? 20 : 24;
            const uint8_t* rw = wt + rl * MM_WT<TY>;
#pragma unroll
            for (int k = 0; k < 4; k++)
                d[k] = *(const uint16_t*)(rw + 2 * BS * k + 2) | ((uint32_t)*(const uint16_t*)(rw + 2 * BS * k + BS + 2) << 16);
        }
    }
    if constexpr (TY == G_Q6K) {
        // pieces to the LDS rows as loaded (unit byte b at sq + b of the quad's row); then the
        // lane reads, from its own row (byte b at sm + b), the dwords the unpacking takes: at 4c
        // and 16 + 4c (two each) of the six 32-byte ql / qh runs, and bytes 192..209 (scales, d),
        // all from the dword-aligned base of the unit's start
        const uint32_t q = (threadIdx.x & 63u) >> 2, pq = threadIdx.x & 3u, kq = (sq + 209) / 16;
#pragma unroll
        for (int l = 0; l < 4; l++)
            if (4 * l + pq <= kq)
                *(u32x4*)(wt + q * 240 + 16 * (4 * l + pq)) = u32x4{s[4 * l], s[4 * l + 1], s[4 * l + 2], s[4 * l + 3]};
        const uint8_t* a = wt + rl * 240 + (sm & ~3u);
#pragma unroll
        for (int k = 0; k < 6; k++) {
            const uint32_t o = k < 4 ? 32 * k : 128 + 32 * (k - 4);
            d[4 * k] = *(const uint32_t*)(a + o + 4 * c);
            d[4 * k + 1] = *(const uint32_t*)(a + o + 4 * c + 4);
            d[4 * k + 2] = *(const uint32_t*)(a + o + 16 + 4 * c);
            d[4 * k + 3] = *(const uint32_t*)(a + o + 20 + 4 * c);
        }
#pragma unroll
        for (int k = 0; k < 5; k++) d[24 + k] = *(const uint32_t*)(a + 192 + 4 * k);
    }
    if constexpr (TY == G_Q4K || TY == G_Q5K) {
        constexpr uint32_t NP = MM_UB<TY> / 16, QP = TY == G_Q4K ? 1 : 3;  // pieces; first qs piece
        const uint32_t q = (threadIdx.x & 63u) >> 2, pq = threadIdx.x & 3u, fq = (q >> 2) & 3u;
#pragma unroll
        for (int l = 0; l < 3; l++)
            if (4 * l + pq < NP)  // (the last load's repeats of the unit's last piece stay out)
                *(u32x4*)(wt + q * MM_WT<TY> + 16 * ((4 * l + pq) ^ fq)) = u32x4{s[4 * l], s[4 * l + 1], s[4 * l + 2], s[4 * l + 3]};
        const uint8_t* rw = wt + rl * MM_WT<TY>;
        const uint32_t fr = (rl >> 2) & 3u;
        const u32x4 h = *(const u32x4*)(rw + 16 * fr);
        d[0] = h[0]; d[1] = h[1]; d[2] = h[2]; d[3] = h[3];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const u32x2 v = *(const u32x2*)(rw + 16 * ((QP + 2 * k + (c >> 1)) ^ fr) + 8 * (c & 1));
            d[4 + 2 * k] = v[0];
            d[5 + 2 * k] = v[1];
        }
        if constexpr (TY == G_Q5K) {
            const u32x2 v = *(const u32x2*)(rw + 16 * ((1 + (c >> 1)) ^ fr) + 8 * (c & 1));
            d[12] = v[0];
            d[13] = v[1];
        }
    }
}

// Max over the wave of unsigned values, in every lane (DPP rotations within 16 lanes, then
// swaps of 16 and 32: no LDS).
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t x) {
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x128, 0xf, 0xf, false));  // row_ror:8
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x124, 0xf, 0xf, false));  // row_ror:4
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x122, 0xf, 0xf, false));  // row_ror:2
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x121, 0xf, 0xf, false));  // row_ror:1
    const auto r16 = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    x = max(r16[0], r16[1]);
    const auto r32 = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return max(r32[0], r32[1]);
}
// The power of two that puts the largest |x| of a unit (four columns a lane) in [2^14, 2^15),
// and its inverse; an infinity or NaN in x stays one, and its unit takes the scale of the largest
// finite numbers. Units below 2^-112 take 2^126 (a zero stays zero). Bits of |x| compare as |x| does.
__device__ __forceinline__ void unit_scale(const float (&x)[4], float& s, float& inv) {
    uint32_t m = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) m = max(m, __float_as_uint(x[e]) & 0x7fffffffu);
    const uint32_t e = min(max(__builtin_amdgcn_readfirstlane(wave_max_u32(m)) >> 23, 15u), 254u);
    s = __uint_as_float((268u - e) << 23);
    inv = __uint_as_float((e - 14u) << 23);
}
// Four columns' hi and lo parts, scaled, in the order of e (x s is exact, so lo's FMA gives
// x s - hi, at most 8). ORDER: tl_order. F16 weights: lo of an infinite x is finite, not
// inf - inf, so the products are IEEE's, as over one row; the block formats' are NaN.
constexpr float MM_LO = 4096.0f, MM_LO_INV = 1.0f / 4096.0f;
template <int ORDER>
__device__ __forceinline__ void hi_lo(const float (&x)[4], float s, half4& h, half4& l) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int e = 0; e < 4; e += 2) {
        const half2 hv = __builtin_convertvector((f32x2{x[e] * s, x[e + 1] * s}), half2);
        const float k = ORDER == 2 ? 1.0f : MM_LO;
        float r[2] = {k * __builtin_fmaf(x[e], s, -(float)hv[0]), k * __builtin_fmaf(x[e + 1], s, -(float)hv[1])};
        if constexpr (ORDER == 0)  // (of NaN, med3 gives a bound)
            for (float& v : r) v = __builtin_amdgcn_fmed3f(v, -8.0f * MM_LO, 8.0f * MM_LO);
        const half2 lv = __builtin_convertvector((f32x2{r[0], r[1]}), half2);
        h[e] = hv[0]; h[e + 1] = hv[1];
        l[e] = lv[0]; l[e + 1] = lv[1];
    }
}
// The sum of a group of 32 columns over its 8 lanes, of hi + lo as they are: what x lost then meets
// a weight a q + b, not a q alone.
__device__ __forceinline__ float group_sum(half4 h, half4 l) {
    float x[4];
#pragma unroll
    for (int e = 0; e < 4; e++) x[e] = __builtin_fmaf(MM_LO_INV, (float)l[e], (float)h[e]);
    float sg = ((x[0] + x[1]) + x[2]) + x[3];
    // DPP moves (lanes i ^ 1, i ^ 2, 7 - i of eight): no LDS.
    sg += __uint_as_float(__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(sg), 0xb1, 0xf, 0xf, false));
    sg += __uint_as_float(__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(sg), 0x4e, 0xf, 0xf, false));
    sg += __uint_as_float(__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(sg), 0x141, 0xf, 0xf, false));
    return sg;
}
// A group's sum of x s / 32 in three parts; SCALED (K-quants, whose m's are small integers): the
// last two times 2^12, over m's times 2^-12.
template <bool SCALED>
__device__ __forceinline__ void sum_parts(float sg, f16 (&p)[3]) {
    float r = sg * 0.03125f;
    p[0] = (f16)r;
    r = (r - (float)p[0]) * (SCALED ? MM_LO : 1.0f);
    p[1] = (f16)r;
    p[2] = (f16)(r - (float)p[1]);
}
// What a unit's groups share: the scale factors and packed scale bytes (K-quants), the b
// factor over x's scale and the eight groups' m's as f16.
struct MMUnit {
    float dl = 0.0f, bl = 0.0f;
    uint32_t scA = 0, scB = 0, mnA = 0, mnB = 0;
};
// The m bytes of a unit (K-quants) as f16 values times k, in group order: (1024 + m) k - 1024 k,
// exact for the k of lane c's part of the sums (1, or 2^-12 for the second and third).
__device__ __forceinline__ f16 mins_scale(uint32_t c) { return c == 0 ? (f16)1.0f : (f16)MM_LO_INV; }
__device__ __forceinline__ half8 mins_f16(uint32_t a, uint32_t b, f16 k) {
    const half2 k2 = half2{k, k}, o = k2 * half2{(f16)-1024.0f, (f16)-1024.0f};
    auto two = [&](uint32_t v, uint32_t sel) {
        return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(half2, __builtin_amdgcn_perm(0x64646464u, v, sel)), k2, o));
    };
    return __builtin_bit_cast(half8, u32x4{two(a, 0x04010400u), two(a, 0x04030402u), two(b, 0x04010400u), two(b, 0x04030402u)});
}

template <uint32_t TY>
__device__ __forceinline__ MMUnit mm_unit(const uint32_t (&d)[MWD<TY>]) {
    MMUnit m;
    if constexpr (TY == G_Q4K || TY == G_Q5K) {
        // scale and min bytes of sub-blocks 0..3 and 4..7 (6 bits each, quant.rs:136-146)
        const uint32_t s0 = d[1], s1 = d[2], s2 = d[3];
        m.scA = s0 & 0x3f3f3f3fu;
        m.scB = (s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u);
        m.mnA = s1 & 0x3f3f3f3fu;
        m.mnB = ((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u);
        m.dl = h2f(d[0] & 0xffffu);
        m.bl = -32.0f * h2f(d[0] >> 16);
    } else if constexpr (TY == G_Q4_1 || TY == G_Q5_1) {
        m.bl = 32.0f;
    }
    return m;
}

// Group j of a loaded unit for lane c: B operand(s) and a. Q6K gives its
// two halves' four weights q4[0], q4[1] and a0, a1.
template <uint32_t TY>
__device__ __forceinline__ void mm_group(const uint32_t (&d)[MWD<TY>], const MMUnit& m, const uint8_t* unit_base,
                                         const uint8_t* rw, int j, uint32_t c, half8& q, half4 (&q4)[2],
                                         float& a0, float& a1) {
    if constexpr (TY == G_F16) {  // weights 8c .. 8c + 7 in order (x staged unpermuted)
        q = __builtin_bit_cast(half8, u32x4{d[4 * j], d[4 * j + 1], d[4 * j + 2], d[4 * j + 3]});
    } else if constexpr (TY == G_Q8_0) {  // from the lane's LDS row rw (the unit, 16-aligned)
        const uint32_t b = 34 * j + 2 + 8 * c, a = b & ~3u, sh = b & 3u;  // qs bytes 8c .. of block j
        const uint32_t w[3] = {*(const uint32_t*)(rw + a), *(const uint32_t*)(rw + a + 4),
                               *(const uint32_t*)(rw + a + 4 + 2 * sh)};
        const uint32_t w0 = __builtin_amdgcn_alignbyte(w[1], w[0], sh), w1 = __builtin_amdgcn_alignbyte(w[2], w[1], sh);
        q = bytes8_f16(w0 ^ 0x80808080u, w1 ^ 0x80808080u, half2{(f16)1152.0f, (f16)1152.0f});
        a0 = h2f(*(const uint16_t*)(rw + 34 * j));
    } else if constexpr (TY == G_Q4_0 || TY == G_Q5_0) {
        // from the lane's LDS row rw; lanes 0, 1: low nibbles, lanes 2, 3: high nibbles
        // (weights 16 ..), as q - 8 (Q4_0) or, with qh byte c as bit 4, q - 16 (Q5_0)
        constexpr uint32_t BS = TY == G_Q4_0 ? 18 : 22, QS = TY == G_Q4_0 ? 2 : 6;
        const uint32_t b = BS * j + QS + 8 * (c & 1), a = b & ~3u, sh = b & 3u;
        const uint32_t w[3] = {*(const uint32_t*)(rw + a), *(const uint32_t*)(rw + a + 4),
                               *(const uint32_t*)(rw + a + 4 + 2 * sh)};
        uint32_t w0 = __builtin_amdgcn_alignbyte(w[1], w[0], sh), w1 = __builtin_amdgcn_alignbyte(w[2], w[1], sh);
        const uint32_t ns = c < 2 ? 0u : 4u;
        if constexpr (TY == G_Q4_0) {
            q = fields8(w0 >> ns, w1 >> ns, 0x000f000fu, half2{(f16)1032.0f, (f16)1032.0f});
        } else {
            const uint32_t qh = *(const uint8_t*)(rw + BS * j + 2 + c);  // bit 4 of weights 8c ..
            w0 = ((w0 >> ns) & 0x0f0f0f0fu) | bit4_spread(qh & 15u);
            w1 = ((w1 >> ns) & 0x0f0f0f0fu) | bit4_spread(qh >> 4);
            q = bytes8_f16(w0, w1, half2{(f16)1040.0f, (f16)1040.0f});
        }
        a0 = h2f(*(const uint16_t*)(rw + BS * j));
    } else if constexpr (TY == G_Q4_1 || TY == G_Q5_1) {  // from the lane's LDS row rw
        constexpr uint32_t BS = TY == G_Q4_1 ? 20 : 24, QS = TY == G_Q4_1 ? 4 : 8;
        const uint8_t* g = rw + BS * j;
        const uint32_t x0 = *(const uint32_t*)(g + QS + 8 * (c & 1)), x1 = *(const uint32_t*)(g + QS + 8 * (c & 1) + 4);
        const uint32_t ns = c < 2 ? 0u : 4u;
        if constexpr (TY == G_Q4_1) {
            q = fields8(x0 >> ns, x1 >> ns, 0x000f000fu, half2{(f16)1024.0f, (f16)1024.0f});
        } else {
            const uint32_t qh = g[4 + c];  // qh byte c
            const uint32_t w0 = ((x0 >> ns) & 0x0f0f0f0fu) | bit4_spread(qh & 15u);
            const uint32_t w1 = ((x1 >> ns) & 0x0f0f0f0fu) | bit4_spread(qh >> 4);
            q = bytes8_f16(w0, w1, half2{(f16)1024.0f, (f16)1024.0f});
        }
        a0 = h2f(*(const uint16_t*)g);
    } else if constexpr (TY == G_Q4K || TY == G_Q5K) {
        const int k = j / 2, hi = j % 2;
        const uint32_t v0 = d[4 + 2 * k], v1 = d[5 + 2 * k];
        // B = q sc_j (an f16 integer): the sub-block scale rides in the unpacking FMA, so the
        // unit's eight MFMAs chain through one accumulator and d scales the unit once.
        // (sc_j, sc_j) from its byte under the exponent of 1024: (1024 + sc) s - 1024 s, with
        // s = 1/16 for Q4K's high nibbles, which stay in place (16 q).
        const uint32_t b = (uint32_t)(j % 4);
        const half2 e = __builtin_bit_cast(half2, __builtin_amdgcn_perm(0x64646464u, j < 4 ? m.scA : m.scB,
                                                                        0x04000400u | b | (b << 16)));
        const f16 s16 = (TY == G_Q4K && hi) ? (f16)0.0625f : (f16)1.0f;
        const half2 c1 = __builtin_elementwise_fma(e, half2{s16, s16}, half2{(f16)-1024.0f * s16, (f16)-1024.0f * s16});
        const half2 c2 = c1 * half2{(f16)-1024.0f, (f16)-1024.0f};
        if constexpr (TY == G_Q4K) {
            const uint32_t mk = hi ? 0x00f000f0u : 0x000f000fu;
            q = __builtin_bit_cast(half8, u32x4{field_pair_sc(v0, mk, c1, c2), field_pair_sc(v0 >> 8, mk, c1, c2),
                                                field_pair_sc(v1, mk, c1, c2), field_pair_sc(v1 >> 8, mk, c1, c2)});
        } else {  // bit j of qh byte t is bit 4 of weight t
            const uint32_t h0 = d[12] >> j, h1 = d[13] >> j;
            const uint32_t n0 = hi ? v0 >> 4 : v0, n1 = hi ? v1 >> 4 : v1;
            const uint32_t m4 = 0x000f000fu, b4 = 0x00010001u;
            q = __builtin_bit_cast(half8, u32x4{field_pair_sc(n0, m4, c1, c2, (h0 & b4) << 4),
                                                field_pair_sc(n0 >> 8, m4, c1, c2, ((h0 >> 8) & b4) << 4),
                                                field_pair_sc(n1, m4, c1, c2, (h1 & b4) << 4),
                                                field_pair_sc(n1 >> 8, m4, c1, c2, ((h1 >> 8) & b4) << 4)});
        }
    } else {  // Q6K
        const int hh = j / 4, qr = j % 4, s = qr & 1;
        const uint32_t sh = (uint32_t)((uintptr_t)unit_base & 3u);
        // lane c: weights 4c .. 4c + 3 (half 0) and 16 + 4c .. (half 1) of the group
        const uint32_t* L = &d[4 * (2 * hh + s)];
        const uint32_t* H = &d[4 * (4 + hh)];
        const uint32_t l0 = __builtin_amdgcn_alignbyte(L[1], L[0], sh), l1 = __builtin_amdgcn_alignbyte(L[3], L[2], sh);
        const uint32_t h0 = __builtin_amdgcn_alignbyte(H[1], H[0], sh), h1 = __builtin_amdgcn_alignbyte(H[3], H[2], sh);
        const uint32_t ns = qr < 2 ? 0u : 4u;
        const uint32_t v0 = ((l0 >> ns) & 0x0f0f0f0fu) | (((h0 >> (2 * qr)) & 0x03030303u) << 4);
        const uint32_t v1 = ((l1 >> ns) & 0x0f0f0f0fu) | (((h1 >> (2 * qr)) & 0x03030303u) << 4);
        const half2 o = half2{(f16)1056.0f, (f16)1056.0f};
        q4[0] = __builtin_bit_cast(half4, bytes_f16(v0, o));
        q4[1] = __builtin_bit_cast(half4, bytes_f16(v1, o));
        // scales (int8) 8 hh + 2 qr and + 1, d: bytes 192 .. 209 of the block
        const uint32_t sw = __builtin_amdgcn_alignbyte(d[25 + hh * 2 + (qr >> 1)], d[24 + hh * 2 + (qr >> 1)], sh);
        const uint32_t sp = sw >> (16 * (qr & 1));  // bytes 2 qr, 2 qr + 1 of the 4-byte window
        const uint32_t dw = __builtin_amdgcn_alignbyte(d[28], d[28], sh) & 0xffffu;  // d: bytes 208, 209
        const float dd = h2f(dw);
        a0 = dd * (float)(int8_t)(uint8_t)(sp & 255u);
        a1 = dd * (float)(int8_t)(uint8_t)((sp >> 8) & 255u);
    }
}

struct MMParams {
    const uint8_t* w;
    const float* x;
    float* out;
    float* part;    // [ks][npad][rows]: parallel splits' partials
    uint32_t* cnt;  // [tiles]: arrivals of a tile's parallel splits (zero between calls)
    uint32_t rows, cols, n, npad, row_bytes, units, ks, par;
};

// NI: input rows a workgroup, 8 (two workgroups a CU) or 16 (one, for batches of 9 to 16:
// each weight unpacked once for all of them).
template <uint32_t TY, int NI>
__global__ __launch_bounds__(64 * MM_W<TY>, NI == 16 ? 2 : MM_W<TY> / 2) void k_matmul_mm(const MMParams p) {
    constexpr bool SUM = mm_sum<TY>(), KP = TY != G_F16, UT = TY == G_Q4K || TY == G_Q5K || TY == G_F16;
    constexpr int PF = MM_PF<TY>, W = MM_W<TY>, NT = 64 * W;
    constexpr uint32_t XS = MM_XS<TY>;
    // hi of the NI inputs, then lo (Q6K: an input's row holds each four columns' hi and lo
    // together, 16 bytes; rows XR apart).
    constexpr uint32_t XR = TY == G_Q6K ? 2 * MM_K<TY> * 256 + 16 : XS;
    __shared__ __attribute__((aligned(16))) f16 xs[2 * NI * XS];
    __shared__ __attribute__((aligned(16))) float isc[MM_K<TY> * NI];
    __shared__ __attribute__((aligned(16))) f16 ss[SUM ? MM_K<TY> * NI * 32 : 4];
    constexpr bool KQ = MM_LDSP<TY>;  // units pass through LDS (mm_fix)
    __shared__ __attribute__((aligned(16))) uint8_t wtb[KQ ? W * 16 * MM_WT<TY> : 16];
    __shared__ uint32_t last;
    static_assert(XR <= 2 * XS, "Q6K's rows fit");
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t c = lane >> 4, rl = lane & 15;
    const uint32_t r0 = blockIdx.x * (16 * W) + 16 * w, r = r0 + rl, i0 = blockIdx.y * NI;
    const bool live = r0 < p.rows;  // the wave has rows
    const f16 mk = mins_scale(c);
    // the rows a lane loads: its matrix-core row (mrowp), or (KQ) its lane quad's
    const uint8_t* mrowp = p.w + (size_t)min(r, p.rows - 1) * p.row_bytes;
    const uint8_t* rowp = KQ ? p.w + (size_t)min(r0 + (lane >> 2), p.rows - 1) * p.row_bytes : mrowp;
    uint8_t* wt = wtb + (KQ ? w * 16 * MM_WT<TY> : 0);
    const uint32_t kz0 = p.par ? blockIdx.z : 0, kz1 = p.par ? blockIdx.z + 1 : p.ks;
    float tot[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (SUM)  // the last quarter of the b terms' A rows stays 0
        for (uint32_t q = tid; q < MM_K<TY> * NI; q += NT) *(half8*)&ss[32 * q + 24] = half8{};
    for (uint32_t kz = kz0; kz < kz1; kz++) {
        const uint32_t ua = kz * p.units / p.ks, nu = (kz + 1) * p.units / p.ks - ua;
        // Every step loads one unit (past the range's end its last unit again), so the loads
        // outstanding at each use are the same and the compiler's waits stay partial.
        uint32_t pk[PF][MW<TY>];
        if (live) {
#pragma unroll
            for (int f = 0; f < PF; f++) mm_load<TY>(rowp, ua + min((uint32_t)f, nu - 1), c, pk[f]);
        }
        if (kz != kz0) __syncthreads();  // every wave is done with the previous split's x
        // Stage x, an input row a wave and a unit (64 float4s, consecutive lanes) a load, as scaled
        // hi and lo in the lanes' k order (within each 8 columns: 0, 2, 1, 3, 4, 6, 5, 7, so a
        // float4's four values stay together); (SUM) a group's sum over the 8 lanes that hold it,
        // in a fixed tree.
        constexpr uint32_t XB = 4;  // loads in flight a thread
        // The scales of four units side by side (one after another, each waits for its moves between
        // lanes), whether the range has four or not: Q4K 14336 x 4096 at 2 / 8 rows 13.7 -> 13.05 and
        // 14.7 -> 14.15 us, Q4_0 14.9 -> 14.5 and 15.3 -> 14.7. Not F16, Q8_0 and Q6K, whose short
        // ranges lost (Q8_0 3584 x 3584 at 8 rows 10.75 -> 11.0).
        constexpr bool AHEAD = TY != G_F16 && TY != G_Q8_0 && TY != G_Q6K;
        // (Inputs past the batch are left as they are: their D rows are not used.)
        const uint32_t ni = min((uint32_t)NI, p.n - i0);
        for (uint32_t i = w; i < ni; i += W) {
            const float* xrow = p.x + (size_t)(i0 + i) * p.cols + (size_t)ua * 256 + 4 * lane;
            for (uint32_t v0 = 0; v0 < nu; v0 += XB) {
                float4 v[XB];
#pragma unroll
                for (uint32_t t = 0; t < XB; t++) v[t] = *(const float4*)(xrow + 256 * min(v0 + t, nu - 1));
                float sc[XB], inv[XB];
                auto scale = [&](uint32_t t) {
                    const float x4[4] = {v[t].x, v[t].y, v[t].z, v[t].w};
                    unit_scale(x4, sc[t], inv[t]);
                };
                if constexpr (AHEAD)
#pragma unroll
                    for (uint32_t t = 0; t < XB; t++) scale(t);
#pragma unroll
                for (uint32_t t = 0; t < XB; t++) {
                    const uint32_t lu = v0 + t, cq = 64 * lu + lane;
                    if (lu >= nu) break;
                    const float x4[4] = {v[t].x, v[t].y, v[t].z, v[t].w};
                    if constexpr (!AHEAD) scale(t);
                    if (lane == 0) isc[lu * NI + i] = inv[t];
                    const float xs4[4] = {x4[0], KP ? x4[2] : x4[1], KP ? x4[1] : x4[2], x4[3]};
                    half4 h, l;
                    hi_lo<tl_order<TY>()>(xs4, sc[t], h, l);
                    if constexpr (SUM) {
                        const float sg = group_sum(h, l);
                        if ((lane & 7) == 0) {
                            f16 sp[3];
                            sum_parts<TY == G_Q4K || TY == G_Q5K>(sg, sp);
#pragma unroll
                            for (int e = 0; e < 3; e++) ss[(lu * NI + i) * 32 + 8 * e + lane / 8] = sp[e];
                        }
                    }
                    if constexpr (TY == G_Q6K) {
                        *(half8*)&xs[i * XR + 8 * cq] = __builtin_shufflevector(h, l, 0, 1, 2, 3, 4, 5, 6, 7);
                    } else {
                        *(half4*)&xs[i * XS + 4 * cq] = h;
                        *(half4*)&xs[(NI + i) * XS + 4 * cq] = l;
                    }
                }
            }
        }
        __syncthreads();
        f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (live) {
            const uint32_t ra = rl & (NI - 1u);  // the lane's A row
            for (uint32_t u0 = 0; u0 < nu; u0 += PF) {
#pragma unroll
                for (int f = 0; f < PF; f++) {
                    const uint32_t lu = u0 + f;
                    if (lu < nu) {
                        const uint8_t* ub = mrowp + (size_t)(ua + lu) * MM_UB<TY>;  // the lane's row's unit
                        const uint8_t* qb = rowp + (size_t)(ua + lu) * MM_UB<TY>;   // its lane quad's
                        uint32_t dd[MWD<TY>];
                        mm_fix<TY>(pk[f], dd, wt, c, rl, (uint32_t)((uintptr_t)qb & 15u), (uint32_t)((uintptr_t)ub & 15u));
                        const MMUnit m = mm_unit<TY>(dd);
                        const f32x4 z4 = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                        f32x4 t4 = z4, t5 = z4;  // hi and lo apart (NI 8: in lanes c < 2 and c >= 2 of t4)
#pragma unroll
                        for (int j = 0; j < 8; j++) {
                            const uint32_t col = lu * 256 + 32 * j;
                            half8 q;
                            half4 qh[2];
                            float a0 = 0.0f, a1 = 0.0f;
                            mm_group<TY>(dd, m, ub, wt + rl * MM_WT<TY>, j, c, q, qh, a0, a1);
                            if constexpr (TY == G_Q6K) {
                                const half8 x0 = *(const half8*)&xs[ra * XR + 2 * col + 8 * c];
                                const half8 x1 = *(const half8*)&xs[ra * XR + 2 * col + 32 + 8 * c];
                                const f32x4 d0 = mfma16(x0, __builtin_shufflevector(qh[0], qh[0], 0, 1, 2, 3, 4, 5, 6, 7), z4);
                                const f32x4 d1 = mfma16(x1, __builtin_shufflevector(qh[1], qh[1], 0, 1, 2, 3, 4, 5, 6, 7), z4);
#pragma unroll
                                for (int i = 0; i < 4; i++) t4[i] = __builtin_fmaf(a1, d1[i], __builtin_fmaf(a0, d0[i], t4[i]));
                            } else {
                                const half8 xh = *(const half8*)&xs[rl * XS + col + 8 * c];
                                half8 xo;
                                if constexpr (NI == 16) xo = *(const half8*)&xs[(16 + rl) * XS + col + 8 * c];
                                if constexpr (UT) {
                                    t4 = mfma16(xh, q, t4);
                                    if constexpr (NI == 16) t5 = mfma16(xo, q, t5);
                                } else {
                                    const f32x4 dv = mfma16(xh, q, z4);
#pragma unroll
                                    for (int i = 0; i < 4; i++) t4[i] = __builtin_fmaf(a0, dv[i], t4[i]);
                                    if constexpr (NI == 16) {
                                        const f32x4 dw = mfma16(xo, q, z4);
#pragma unroll
                                        for (int i = 0; i < 4; i++) t5[i] = __builtin_fmaf(a0, dw[i], t5[i]);
                                    }
                                }
                            }
                        }
                        if constexpr (TY != G_Q6K) {  // hi + lo
                            if constexpr (NI == 16) {
#pragma unroll
                                for (int i = 0; i < 4; i++) t4[i] = __builtin_fmaf(MM_LO_INV, t5[i], t4[i]);
                            } else {
#pragma unroll
                                for (int i = 0; i < 4; i++) {
                                    const auto r2 = __builtin_amdgcn_permlane32_swap(__float_as_uint(t4[i]), __float_as_uint(t4[i]), false, false);
                                    t4[i] = __builtin_fmaf(MM_LO_INV, __uint_as_float(r2[1]), __uint_as_float(r2[0]));
                                }
                            }
                        }
                        const float4 is = *(const float4*)&isc[lu * NI + 4 * (c & (NI / 4 - 1u))];
                        const float i4[4] = {is.x, is.y, is.z, is.w};
                        if constexpr (TY == G_Q4K || TY == G_Q5K) t4 *= m.dl;
                        if constexpr (SUM) {
                            half8 mv;
                            if constexpr (TY == G_Q4K || TY == G_Q5K) mv = mins_f16(m.mnA, m.mnB, mk);
                            else mv = __builtin_bit_cast(half8, u32x4{dd[0], dd[1], dd[2], dd[3]});
                            const f32x4 tb = mfma16(*(const half8*)&ss[(lu * NI + ra) * 32 + 8 * c], mv, z4);
#pragma unroll
                            for (int i = 0; i < 4; i++) t4[i] = __builtin_fmaf(m.bl, tb[i], t4[i]);
                        }
#pragma unroll
                        for (int i = 0; i < 4; i++) acc[i] = __builtin_fmaf(i4[i], t4[i], acc[i]);
                    }
                    // the unit's registers are free: load into them directly (a load hoisted
                    // above their last use would land in other registers and wait to be copied)
                    __builtin_amdgcn_sched_barrier(0);
                    mm_load<TY>(rowp, ua + min(lu + PF, nu - 1), c, pk[f]);
                }
            }
        }
        // the split's partial (input 4c + i in lanes c < NI / 4); then the splits in order
#pragma unroll
        for (int i = 0; i < 4; i++) tot[i] = kz == kz0 ? acc[i] : tot[i] + acc[i];
    }
    if (!p.par) {
        if (c < NI / 4 && r < p.rows) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (i0 + 4 * c + i < p.n) p.out[(size_t)(i0 + 4 * c + i) * p.rows + r] = tot[i];
        }
        return;
    }
    // Parallel splits: the partial to device memory (write-through stores), then the tile's
    // arrival count; the last workgroup of the tile adds the partials in split order.
    if (c < NI / 4 && r < p.rows) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            __hip_atomic_store(&p.part[((size_t)blockIdx.z * p.npad + i0 + 4 * c + i) * p.rows + r], tot[i],
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __builtin_amdgcn_s_waitcnt(0);  // this thread's stores are done
    __syncthreads();
    const uint32_t tile = blockIdx.y * gridDim.x + blockIdx.x;
    if (tid == 0) {
        const uint32_t old = __hip_atomic_fetch_add(&p.cnt[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = old == p.ks - 1;
    }
    __syncthreads();
    if (!last) return;
    // The tile's NI x 16 W outputs, two a thread and pass; eight splits' loads in flight at a time.
    const size_t stride = (size_t)p.npad * p.rows;
    for (uint32_t q = 0; q < NI * 16 * W; q += 2 * NT) {
        float sum[2] = {0.0f, 0.0f};
        bool ok[2];
        const float* src[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t e = q + tid + h * NT, rr = blockIdx.x * (16 * W) + e % (16 * W), in = i0 + e / (16 * W);
            ok[h] = rr < p.rows && in < p.n;
            src[h] = p.part + (size_t)min(in, p.npad - 1) * p.rows + min(rr, p.rows - 1);
        }
        for (uint32_t k0 = 0; k0 < p.ks; k0 += 8) {
            float v[2][8];
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int t = 0; t < 8; t++)
                    v[h][t] = k0 + t < p.ks ? __hip_atomic_load(src[h] + (k0 + t) * stride, __ATOMIC_RELAXED,
                                                                 __HIP_MEMORY_SCOPE_AGENT)
                                            : 0.0f;
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int t = 0; t < 8; t++)
                    if (k0 + t < p.ks) sum[h] = k0 + t == 0 ? v[h][t] : sum[h] + v[h][t];
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t e = q + tid + h * NT, rr = blockIdx.x * (16 * W) + e % (16 * W), in = i0 + e / (16 * W);
            if (ok[h]) p.out[(size_t)in * p.rows + rr] = sum[h];
        }
    }
    if (tid == 0) __hip_atomic_store(&p.cnt[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One input row (decode) of the block formats, cols a multiple of 256: a workgroup is 16 weight
// rows, its W waves take the units in turn (one loaded ahead; ONE: a wave has one unit at most),
// each staging its own unit's x and weights in its own LDS without a barrier. A unit's end and
// the units' sum are in 64 bits (a few operations a unit), so the error stays at or below the
// vector-unit pass's, whose f32 chains were shorter. Every A row 0 .. 7 is x's hi
// and 8 .. 15 its lo (Q6K: both together), so staging is one row and the reads are broadcasts.
// The vector-unit pass (k_matmul) held 1.75 waves a SIMD on this work, each waiting for a column
// tile and then converting and multiplying it; here the products go to the matrix cores and the
// waves are seven a SIMD, which leaves the unpacking (Q6K) and the loads (the others).
// One row, us a call, k_matmul -> here, over 470 to 900 MB of matrices in turn (weights from HBM): Q4K
// 14336 x 4096 15.3 -> 12.6, 4096 x 14336 19.8 -> 12.3, 1024 x 4096 7.0 -> 4.4; Q6K 22.9 -> 18.5, 27.1 ->
// 17.0, 9.1 -> 5.5; Q8_0 21.6 -> 15.3, 24.3 -> 15.6, 8.1 -> 4.8; over six matrices, which the 256 MB
// cache holds for Q4K, 14.1 -> 11.3, 18.0 -> 11.0, 5.9 -> 3.9. 32 rows a workgroup (x staged once for
// both) were 6% faster at Q4K 28672 x 8192 and 9-18% slower for Q8_0 and Q4_0. Error against 64 bits
// at 4096 columns: Q4_0 2.6e-7 -> 0.8e-7, Q8_0 1.1 -> 0.8, Q4K 1.7 -> 1.4, Q5K 1.7 -> 1.5, Q6K 2.3 -> 1.0.
constexpr uint32_t ROW_UNITS = 256;  // units whose sums fit the workgroup's LDS

template <uint32_t TY, int W, bool ONE>
__global__ __launch_bounds__(64 * W) void k_matmul_row(const MMParams p) {
    constexpr bool SUM = mm_sum<TY>(), UT = TY == G_Q4K || TY == G_Q5K;
    static_assert(MM_LDSP<TY>, "block formats");
    constexpr uint32_t XL = 288;  // halves from hi to lo: other banks
    __shared__ __attribute__((aligned(16))) f16 xs[W][XL + 256];
    __shared__ __attribute__((aligned(16))) uint8_t wtb[W][16 * MM_WT<TY>];
    __shared__ __attribute__((aligned(16))) f16 ss[W][SUM ? 32 : 8];
    extern __shared__ __attribute__((aligned(16))) double ps[];  // [units][16], then [units] inverse scales
    float* isc = (float*)(ps + p.units * 16);
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t c = lane >> 4, rl = lane & 15;
    const uint32_t r0 = blockIdx.x * 16;
    // the lane's matrix-core row and its lane quad's
    const uint8_t* mrow = p.w + (size_t)min(r0 + rl, p.rows - 1) * p.row_bytes;
    const uint8_t* qrow = p.w + (size_t)min(r0 + (lane >> 2), p.rows - 1) * p.row_bytes;
    uint8_t* wt = wtb[w];
    const f16 mk = mins_scale(c);
    // LDS written and read by one wave only: in order, no barrier.
    auto own = [&]() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
    if constexpr (SUM)
        if (lane == 0) *(half8*)&ss[w][24] = half8{};
    constexpr int PF = ONE ? 1 : 2;
    uint32_t pk[PF][MW<TY>];
    float4 xv[PF];
    // Past the wave's last unit the loads are of the first row's first unit, the same few lines for
    // every wave, so that each use waits for a fixed number of loads.
    auto load = [&](uint32_t u, uint32_t (&d)[MW<TY>], float4& x) {
        const bool in = u < p.units;
        const uint32_t uu = in ? u : 0;
        x = *(const float4*)(p.x + (size_t)uu * 256 + 4 * lane);
        mm_load<TY>(in ? qrow : p.w, uu, c, d);
    };
    load(w, pk[0], xv[0]);
    if constexpr (!ONE) load(w + W, pk[1], xv[1]);
    for (uint32_t u0 = w; u0 < p.units; u0 += PF * W) {
#pragma unroll
        for (int f = 0; f < PF; f++) {
            const uint32_t u = u0 + f * W;
            if (u < p.units) {
                const float x4[4] = {xv[f].x, xv[f].y, xv[f].z, xv[f].w};
                float sc, inv;
                unit_scale(x4, sc, inv);
                if (lane == 0) isc[u] = inv;
                const float xo[4] = {x4[0], x4[2], x4[1], x4[3]};
                half4 h, o;
                hi_lo<tl_order<TY>()>(xo, sc, h, o);
                if constexpr (SUM) {
                    const float sg = group_sum(h, o);
                    if ((lane & 7) == 0) {
                        f16 sp[3];
                        sum_parts<UT>(sg, sp);
#pragma unroll
                        for (int e = 0; e < 3; e++) ss[w][8 * e + lane / 8] = sp[e];
                    }
                }
                if constexpr (TY == G_Q6K) {
                    *(half8*)&xs[w][8 * lane] = __builtin_shufflevector(h, o, 0, 1, 2, 3, 4, 5, 6, 7);
                } else {
                    *(half4*)&xs[w][4 * lane] = h;
                    *(half4*)&xs[w][XL + 4 * lane] = o;
                }
                own();
                const f16* xr = &xs[w][TY == G_Q6K || rl < 8 ? 0 : XL];
                const f32x4 z4 = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                const uint8_t* ub = mrow + (size_t)u * MM_UB<TY>;
                const uint8_t* qb = qrow + (size_t)u * MM_UB<TY>;
                uint32_t dd[MWD<TY>];
                mm_fix<TY>(pk[f], dd, wt, c, rl, (uint32_t)((uintptr_t)qb & 15u), (uint32_t)((uintptr_t)ub & 15u));
                const MMUnit m = mm_unit<TY>(dd);
                f32x4 t4 = z4;
                float s = 0.0f;
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    half8 q;
                    half4 qh[2];
                    float a0 = 0.0f, a1 = 0.0f;
                    mm_group<TY>(dd, m, ub, wt + rl * MM_WT<TY>, j, c, q, qh, a0, a1);
                    if constexpr (TY == G_Q6K) {
                        const half8 x0 = *(const half8*)&xr[64 * j + 8 * c], x1 = *(const half8*)&xr[64 * j + 32 + 8 * c];
                        const f32x4 d0 = mfma16(x0, __builtin_shufflevector(qh[0], qh[0], 0, 1, 2, 3, 4, 5, 6, 7), z4);
                        const f32x4 d1 = mfma16(x1, __builtin_shufflevector(qh[1], qh[1], 0, 1, 2, 3, 4, 5, 6, 7), z4);
                        s = __builtin_fmaf(a1, d1[0], __builtin_fmaf(a0, d0[0], s));
                    } else {
                        const half8 xa = *(const half8*)&xr[32 * j + 8 * c];
                        if constexpr (UT)
                            t4 = mfma16(xa, q, t4);
                        else
                            s = __builtin_fmaf(a0, mfma16(xa, q, z4)[0], s);
                    }
                }
                if constexpr (UT) s = t4[0];
                double sum = s;
                if constexpr (TY != G_Q6K) {  // hi + lo
                    const auto r2 = __builtin_amdgcn_permlane32_swap(__float_as_uint(s), __float_as_uint(s), false, false);
                    sum = __builtin_fma((double)MM_LO_INV, (double)__uint_as_float(r2[1]), (double)__uint_as_float(r2[0]));
                }
                if constexpr (UT) sum *= (double)m.dl;
                if constexpr (SUM) {
                    half8 mv;
                    if constexpr (UT) mv = mins_f16(m.mnA, m.mnB, mk);
                    else mv = __builtin_bit_cast(half8, u32x4{dd[0], dd[1], dd[2], dd[3]});
                    sum = __builtin_fma((double)m.bl, (double)mfma16(*(const half8*)&ss[w][8 * c], mv, z4)[0], sum);
                }
                if (c == 0) ps[u * 16 + rl] = sum;
                own();
            }
            // the unit's registers are free: load into them directly
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (!ONE) load(u + 2 * W, pk[f], xv[f]);
        }
    }
    __syncthreads();
    if (tid >= 16 || r0 + tid >= p.rows) return;
    double tot = 0.0;
    for (uint32_t u = 0; u < p.units; u++) tot = __builtin_fma((double)isc[u], ps[u * 16 + tid], tot);
    p.out[r0 + tid] = (float)tot;
}

// ---------------------------------------------------------------------------------------
// Batched product of many input rows (prompts). k_matmul_mm's workgroups hold 8 input rows,
// so a batch of n unpacks every weight n / 8 times and is bound by that VALU work (512 rows
// of 14336 x 4096 Q4K: 480 us). Here a workgroup of eight waves takes MT input rows x 128
// weight rows and walks its K range in steps of 64 columns (two groups): the step's packed
// weights are loaded by four threads a row (two steps ahead), unpacked once into f16 in LDS
// and read back as the B operands of every input tile; x comes from k_mm_prep as scaled hi
// and lo parts in the operands' order (the conversion once a call instead of once a
// workgroup). Each wave owns TM x TN 16 x 16 output tiles.
//
// Every output element sees k_matmul_mm's operations in k_matmul_mm's order, so an input
// row's bits stay those of the same row in a batch of 2. Formats of 32-weight blocks also
// come here when cols is no multiple of 256 (the last unit is then shorter): those shapes
// have no k_matmul_mm form and took the VALU.
constexpr int TL_NT = 128;       // weight rows a workgroup
constexpr int TL_THREADS = 512;  // eight waves; four threads a weight row

template <uint32_t TY>
constexpr bool tl_kq() {
    return TY == G_Q4K || TY == G_Q5K;
}

// Prepared x of one unit of one input row, a wave: per step 256 bytes, hi of its 64 columns
// then lo (order 2: 16-byte pieces of four columns' hi and lo); the inverse scale; (SUM: 1, or 2
// for the K-quants) the A operand of the b sum x terms. Rows past n and columns past cols are zeros.
template <int ORDER, int SUM>
__global__ __launch_bounds__(256) void k_mm_prep(const float* __restrict__ x, f16* __restrict__ xp,
                                                 float* __restrict__ ip, f16* __restrict__ sp, uint32_t n,
                                                 uint32_t cols, uint32_t npad, uint32_t steps) {
    const uint32_t lane = threadIdx.x & 63u, row = blockIdx.y * 4 + (threadIdx.x >> 6), u = blockIdx.x;
    const uint32_t col = 256 * u + 4 * lane;
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (row < n && col < cols) v = *(const float4*)(x + (size_t)row * cols + col);
    const float x4[4] = {v.x, v.y, v.z, v.w};
    float sc, inv;
    unit_scale(x4, sc, inv);
    const size_t at = (size_t)u * npad + row;
    if (lane == 0) ip[at] = inv;
    const float xo[4] = {v.x, ORDER ? v.z : v.y, ORDER ? v.y : v.z, v.w};
    half4 h, l;
    hi_lo<ORDER>(xo, sc, h, l);
    if constexpr (SUM != 0) {
        const float sg = group_sum(h, l);
        if ((lane & 7u) == 0) {
            f16 p[3];
            sum_parts<SUM == 2>(sg, p);
#pragma unroll
            for (int e = 0; e < 4; e++) sp[at * 32 + 8 * e + lane / 8] = e < 3 ? p[e] : (f16)0.0f;
        }
    }
    const uint32_t step = 4 * u + lane / 16, q = lane % 16;
    if (step >= steps) return;
    f16* dst = xp + ((size_t)step * npad + row) * 128;
    if constexpr (ORDER == 2) {
        *(half8*)(dst + 8 * q) = __builtin_shufflevector(h, l, 0, 1, 2, 3, 4, 5, 6, 7);
    } else {
        *(half4*)(dst + 4 * q) = h;
        *(half4*)(dst + 64 + 4 * q) = l;
    }
}

struct TLParams {
    const uint8_t* w;
    const f16* xp;    // [steps][npad][128]
    const float* ip;  // [units][npad]: inverse scales
    const f16* sp;    // [units][npad][32]: the group sums' parts
    float* out;
    float* part;
    uint32_t* cnt;
    uint32_t rows, n, npad, row_bytes, units, groups, ks, par, nyt;
};

// Bytes at an address that may be 2-byte aligned only (the hardware takes such loads).
template <typename T>
__device__ __forceinline__ T ldu(const uint8_t* p) {
    T v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, 2), sizeof(T));
    return v;
}

// A thread's packed bytes of one step: row r, quarter qd. Groups 2s and 2s + 1 of the row
// are g = 0, 1. K-quants and Q6K: bytes 8 qd .. of each 32-byte run; 32-weight formats and
// F16: half qd & 1 of group qd >> 1. Every byte loaded is used (a load's unused register
// would be taken for something else, which waits for the load).
template <uint32_t TY>
constexpr int TLP = TY == G_F16 ? 8 : TY == G_Q4K ? 2 : TY == G_Q5K ? 4 : TY == G_Q6K ? 6 : 6;
// Load instructions of a step at least.
template <uint32_t TY>
constexpr int TLN = TY == G_Q4K ? 1 : 2;
// A K-quant unit's header: d, dmin and the scale bytes; Q6K's 16 scales and d.
template <uint32_t TY>
constexpr int TLH = tl_kq<TY>() ? 4 : TY == G_Q6K ? 5 : 1;

template <uint32_t TY>
__device__ __forceinline__ void tl_load(const uint8_t* __restrict__ row, uint32_t step, uint32_t qd, uint32_t groups,
                                        uint32_t (&d)[TLP<TY>]) {
    if constexpr (tl_kq<TY>()) {
        const uint8_t* b = row + (size_t)(step / 4) * (TY == G_Q4K ? 144 : 176) + 8 * qd;
        const u32x2 v = *(const u32x2*)(b + (TY == G_Q4K ? 16 : 48) + 32 * (step % 4));
        d[0] = v[0]; d[1] = v[1];
        if constexpr (TY == G_Q5K) {
            const u32x2 q = *(const u32x2*)(b + 16);
            d[2] = q[0]; d[3] = q[1];
        }
    } else if constexpr (TY == G_Q6K) {
        const uint32_t hh = (step % 4) / 2;
        const uint8_t* b = row + (size_t)(step / 4) * 210 + 8 * qd;
        const u32x2 v0 = ldu<u32x2>(b + 64 * hh), v1 = ldu<u32x2>(b + 64 * hh + 32), v2 = ldu<u32x2>(b + 128 + 32 * hh);
        d[0] = v0[0]; d[1] = v0[1];  // group 2c
        d[2] = v1[0]; d[3] = v1[1];  // group 2c + 1
        d[4] = v2[0]; d[5] = v2[1];
    } else {
        const uint32_t g = min(2 * step + (qd >> 1), groups - 1), hf = qd & 1;  // (past the row: its last group)
        if constexpr (TY == G_F16) {
            const u32x4* b = (const u32x4*)(row + (size_t)g * 64 + 32 * hf);
            const u32x4 v0 = b[0], v1 = b[1];
            d[0] = v0[0]; d[1] = v0[1]; d[2] = v0[2]; d[3] = v0[3];
            d[4] = v1[0]; d[5] = v1[1]; d[6] = v1[2]; d[7] = v1[3];
        } else {
            constexpr uint32_t BS = TY == G_Q8_0 ? 34 : TY == G_Q4_0 ? 18 : TY == G_Q4_1 ? 20 : TY == G_Q5_0 ? 22 : 24;
            constexpr uint32_t QS = TY == G_Q8_0 || TY == G_Q4_0 ? 2 : TY == G_Q4_1 ? 4 : TY == G_Q5_0 ? 6 : 8;
            const uint8_t* b = row + (size_t)g * BS;
            const u32x4 v = ldu<u32x4>(b + QS + (TY == G_Q8_0 ? 16 * hf : 0));
            d[0] = v[0]; d[1] = v[1]; d[2] = v[2]; d[3] = v[3];
            d[4] = (TY == G_Q4_1 || TY == G_Q5_1) ? ldu<uint32_t>(b) : (uint32_t)*(const uint16_t*)b;
            if constexpr (TY == G_Q5_0 || TY == G_Q5_1) d[5] = ldu<uint32_t>(b + (TY == G_Q5_0 ? 2 : 4));
        }
    }
}

template <uint32_t TY>
__device__ __forceinline__ void tl_head(const uint8_t* __restrict__ row, uint32_t u, uint32_t (&h)[TLH<TY>]) {
    if constexpr (tl_kq<TY>()) {
        const u32x4 v = *(const u32x4*)(row + (size_t)u * (TY == G_Q4K ? 144 : 176));
        h[0] = v[0]; h[1] = v[1]; h[2] = v[2]; h[3] = v[3];
    } else if constexpr (TY == G_Q6K) {
        const uint8_t* b = row + (size_t)u * 210 + 192;
        const u32x4 v = ldu<u32x4>(b);
        h[0] = v[0]; h[1] = v[1]; h[2] = v[2]; h[3] = v[3];
        h[4] = *(const uint16_t*)(b + 16);
    }
}

// Unpacks a thread's share of a step (its unit's step c) into LDS: its bytes of its row's B
// operands (piece 4 g + c': group g's k slots 8c' ..; Q6K: the four weights of each half of
// lane c'), the group scales (sa), and at a unit's first step the unit's factors: d and b
// (uf) and the eight m's (um). h: the unit's header as loaded (c == 0), kept as m.
template <uint32_t TY, bool FULL, int NT = TL_NT>
__device__ __forceinline__ void tl_stash(const uint32_t (&d)[TLP<TY>], const uint32_t (&h)[TLH<TY>], MMUnit& m,
                                         uint32_t step, uint32_t c, uint32_t r, uint32_t qd, uint32_t groups,
                                         uint8_t* wl, float* sa, float* uf, f16* um) {
    auto at = [&](uint32_t piece) { return wl + r * 128 + 16 * (piece ^ ((r >> 1) & 7u)); };
    auto put = [&](uint32_t piece, half8 v) { *(half8*)at(piece) = v; };
    if constexpr (tl_kq<TY>()) {
        if (c == 0) {
            const uint32_t dd[MWD<TY>] = {h[0], h[1], h[2], h[3]};
            m = mm_unit<TY>(dd);
            if (qd == 0) *(float2*)(uf + 2 * r) = float2{m.dl, m.bl};
            // (the m's over the sums' first part, then over the other two)
            if (qd & 1) *(half8*)(um + 8 * (r + (qd & 2u ? NT : 0))) = mins_f16(m.mnA, m.mnB, mins_scale(qd & 2u));
        }
#pragma unroll
        for (uint32_t hi = 0; hi < 2; hi++) {
            const uint32_t j = 2 * c + hi, sc = ((j < 4 ? m.scA : m.scB) >> (8 * (j & 3u))) & 255u;
            const half2 e = __builtin_bit_cast(half2, sc * 0x00010001u | 0x64006400u);
            const f16 s16 = (TY == G_Q4K && hi) ? (f16)0.0625f : (f16)1.0f;
            const half2 c1 = __builtin_elementwise_fma(e, half2{s16, s16}, half2{(f16)-1024.0f * s16, (f16)-1024.0f * s16});
            const half2 c2 = c1 * half2{(f16)-1024.0f, (f16)-1024.0f};
            const uint32_t v0 = d[0], v1 = d[1];
            if constexpr (TY == G_Q4K) {
                const uint32_t mk = hi ? 0x00f000f0u : 0x000f000fu;
                put(4 * hi + qd, __builtin_bit_cast(half8, u32x4{field_pair_sc(v0, mk, c1, c2), field_pair_sc(v0 >> 8, mk, c1, c2),
                                                                 field_pair_sc(v1, mk, c1, c2), field_pair_sc(v1 >> 8, mk, c1, c2)}));
            } else {
                const uint32_t h0 = d[2] >> j, h1 = d[3] >> j, n0 = hi ? v0 >> 4 : v0, n1 = hi ? v1 >> 4 : v1;
                const uint32_t m4 = 0x000f000fu, b4 = 0x00010001u;
                put(4 * hi + qd, __builtin_bit_cast(half8, u32x4{field_pair_sc(n0, m4, c1, c2, (h0 & b4) << 4),
                                                                 field_pair_sc(n0 >> 8, m4, c1, c2, ((h0 >> 8) & b4) << 4),
                                                                 field_pair_sc(n1, m4, c1, c2, (h1 & b4) << 4),
                                                                 field_pair_sc(n1 >> 8, m4, c1, c2, ((h1 >> 8) & b4) << 4)}));
            }
        }
    } else if constexpr (TY == G_Q6K) {
        // The row's 16 scales, a dword a step, and d.
        if (c == 0) {
            m.scA = h[0];
            m.scB = h[1];
            m.mnA = h[2];
            m.mnB = h[3];
            m.dl = h2f(h[4]);
        }
        const half2 o = half2{(f16)1056.0f, (f16)1056.0f};
#pragma unroll
        for (uint32_t g = 0; g < 2; g++) {
            const uint32_t qr = 2 * (c % 2) + g, ns = (c % 2) * 4;
            const uint32_t v0 = ((d[2 * g] >> ns) & 0x0f0f0f0fu) | (((d[4] >> (2 * qr)) & 0x03030303u) << 4);
            const uint32_t v1 = ((d[2 * g + 1] >> ns) & 0x0f0f0f0fu) | (((d[5] >> (2 * qr)) & 0x03030303u) << 4);
            // weights 8 qd .. 8 qd + 7: half qd >> 1, lanes 2 (qd & 1) and the next
            const uint32_t c2 = 2 * (qd & 1u);
            *(half4*)(at(4 * g + c2) + 8 * (qd >> 1)) = __builtin_bit_cast(half4, bytes_f16(v0, o));
            *(half4*)(at(4 * g + c2 + 1) + 8 * (qd >> 1)) = __builtin_bit_cast(half4, bytes_f16(v1, o));
        }
        const uint32_t sw = c == 0 ? m.scA : c == 1 ? m.scB : c == 2 ? m.mnA : m.mnB;  // the step's four scales
        sa[qd * NT + r] = m.dl * (float)(int8_t)(uint8_t)(sw >> (8 * qd));
    } else {
        const uint32_t gi = qd >> 1, hf = qd & 1, piece = 4 * gi + 2 * hf;
        if constexpr (TY == G_F16) {
            put(piece, __builtin_bit_cast(half8, u32x4{d[0], d[1], d[2], d[3]}));
            put(piece + 1, __builtin_bit_cast(half8, u32x4{d[4], d[5], d[6], d[7]}));
        } else {
            if (hf == 0) sa[gi * NT + r] = h2f(d[4] & 0xffffu);
            if constexpr (TY == G_Q4_1 || TY == G_Q5_1) {
                // m of the step's groups; at the unit's first step 0 for those past the row
                const uint32_t g = 2 * step + gi;
                if (!FULL && c == 0)
#pragma unroll
                    for (uint32_t k = 0; k < 2; k++)
                        if (2 * step + 2 * qd + k >= groups) um[8 * r + 2 * qd + k] = (f16)0.0f;
                if (hf == 1 && g < groups) um[8 * r + (g & 7u)] = __builtin_bit_cast(f16, (uint16_t)(d[4] >> 16));
            }
            if constexpr (TY == G_Q8_0) {
                const half2 o = half2{(f16)1152.0f, (f16)1152.0f};
                put(piece, bytes8_f16(d[0] ^ 0x80808080u, d[1] ^ 0x80808080u, o));
                put(piece + 1, bytes8_f16(d[2] ^ 0x80808080u, d[3] ^ 0x80808080u, o));
            } else {
                const uint32_t ns = 4 * hf;
                constexpr bool FIVE = TY == G_Q5_0 || TY == G_Q5_1;
                const f16 off = TY == G_Q4_0 ? (f16)1032.0f : TY == G_Q5_0 ? (f16)1040.0f : (f16)1024.0f;
#pragma unroll
                for (uint32_t k = 0; k < 2; k++) {
                    if constexpr (FIVE) {
                        const uint32_t qh = (d[5] >> (16 * hf + 8 * k)) & 255u;
                        put(piece + k, bytes8_f16(((d[2 * k] >> ns) & 0x0f0f0f0fu) | bit4_spread(qh & 15u),
                                                  ((d[2 * k + 1] >> ns) & 0x0f0f0f0fu) | bit4_spread(qh >> 4), half2{off, off}));
                    } else {
                        put(piece + k, fields8(d[2 * k] >> ns, d[2 * k + 1] >> ns, 0x000f000fu, half2{off, off}));
                    }
                }
            }
        }
    }
}

// Small batches whose cols is no multiple of 256, in one launch: a workgroup is 16 weight rows x
// 8 input rows, its W waves (four for at most four units: more workgroups then share a CU, else
// eight) take the units in turn, each staging its own unit's x (as k_matmul_mm does) and weights
// (as the tile kernel does) in its own LDS without a barrier, and the units' sums meet in order.
// Bound by latency: Q8_0 4864 x 896 at 2 / 6 / 16 rows 5.3 / 6.2 / 9.2 us (the VALU pass of 8
// rows 7.8 / 14 / 31; the tile kernel and its preparation 13).
// LONG: more units than the workgroup's LDS holds sums of go in stretches (the tile kernel's
// work, but for a call whose scratch cannot be had; the loop over stretches cost the others 2%).
constexpr uint32_t WV_UNITS = 56;

template <uint32_t TY, int W, bool LONG>
__global__ __launch_bounds__(64 * W) void k_matmul_units(const TLParams p, const float* __restrict__ x, uint32_t cols) {
    constexpr bool SUM = mm_sum<TY>(), UT = TY == G_F16;
    constexpr int XS = 264;  // halves an x row
    static_assert(!tl_kq<TY>() && TY != G_Q6K, "formats of 32-weight blocks");
    __shared__ __attribute__((aligned(16))) f16 xs[W][16 * XS];  // inputs' hi, then lo
    __shared__ __attribute__((aligned(16))) uint8_t wl[W][2][16 * 128];
    __shared__ float sa[W][2][UT ? 1 : 2 * 16];
    __shared__ __attribute__((aligned(16))) f16 um[W][SUM ? 8 * 16 : 1];
    __shared__ __attribute__((aligned(16))) f16 ss[W][SUM ? 8 * 32 : 1];
    __shared__ float ps[WV_UNITS][8][16], isc[WV_UNITS][8];
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t c = lane >> 4, l = lane & 15, tr = lane >> 2, qd = lane & 3;
    const uint32_t r0 = blockIdx.x * 16, i0 = blockIdx.y * 8, ni = min(8u, p.n - i0);
    const uint8_t* wrow = p.w + (size_t)min(r0 + tr, p.rows - 1) * p.row_bytes;
    const f32x4 z4 = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const uint32_t nsteps = (p.groups + 1) / 2;
    // LDS written and read by one wave only: in order, no barrier.
    auto own = [&]() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
    if constexpr (SUM)
        if (lane < 8) *(half8*)&ss[w][32 * lane + 24] = half8{};
    auto stretch = [&](uint32_t u0, uint32_t ue) {
        for (uint32_t u = u0 + w; u < ue; u += W) {
            uint32_t pk[4][TLP<TY>], hd[TLH<TY>];
            MMUnit mu;
            const uint32_t ns = min(4u, nsteps - 4 * u);
#pragma unroll
            for (uint32_t s = 0; s < 4; s++) tl_load<TY>(wrow, min(4 * u + s, nsteps - 1), qd, p.groups, pk[s]);
            const uint32_t col = 256 * u + 4 * lane;
            float4 v[8];
#pragma unroll
            for (uint32_t i = 0; i < 8; i++)
                v[i] = *(const float4*)(x + (size_t)(i0 + min(i, ni - 1)) * cols + min(col, cols - 4));
#pragma unroll
            for (uint32_t i = 0; i < 8; i++) {
                if (i >= ni) break;
                const bool in = col < cols;
                const float x4[4] = {in ? v[i].x : 0.0f, in ? v[i].y : 0.0f, in ? v[i].z : 0.0f, in ? v[i].w : 0.0f};
                float sc, inv;
                unit_scale(x4, sc, inv);
                if (lane == 0) isc[u - u0][i] = inv;
                const float xo[4] = {x4[0], UT ? x4[1] : x4[2], UT ? x4[2] : x4[1], x4[3]};
                half4 h, o;
                hi_lo<tl_order<TY>()>(xo, sc, h, o);
                if constexpr (SUM) {
                    const float sg = group_sum(h, o);
                    if ((lane & 7) == 0) {
                        f16 sp[3];
                        sum_parts<false>(sg, sp);
#pragma unroll
                        for (int e = 0; e < 3; e++) ss[w][i * 32 + 8 * e + lane / 8] = sp[e];
                    }
                }
                *(half4*)&xs[w][i * XS + 4 * lane] = h;
                *(half4*)&xs[w][(8 + i) * XS + 4 * lane] = o;
            }
            f32x4 t = z4;  // hi in lanes c < 2, lo in c >= 2
#pragma unroll
            for (uint32_t s = 0; s < 4; s++) {
                if (s >= ns) break;
                tl_stash<TY, false, 16>(pk[s], hd, mu, 4 * u + s, s, tr, qd, p.groups, wl[w][s & 1], sa[w][s & 1], nullptr, um[w]);
                own();
#pragma unroll
                for (uint32_t g = 0; g < 2; g++) {
                    if (8 * u + 2 * s + g >= p.groups) break;
                    const half8 b = *(const half8*)(wl[w][s & 1] + l * 128 + 16 * ((4 * g + c) ^ ((l >> 1) & 7u)));
                    const half8 xa = *(const half8*)&xs[w][l * XS + 64 * s + 32 * g + 8 * c];
                    if constexpr (UT) {
                        t = mfma16(xa, b, t);
                    } else {
                        const f32x4 d = mfma16(xa, b, z4);
                        const float a = sa[w][s & 1][g * 16 + l];
#pragma unroll
                        for (int e = 0; e < 4; e++) t[e] = __builtin_fmaf(a, d[e], t[e]);
                    }
                }
                own();
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const auto r2 = __builtin_amdgcn_permlane32_swap(__float_as_uint(t[e]), __float_as_uint(t[e]), false, false);
                t[e] = __builtin_fmaf(MM_LO_INV, __uint_as_float(r2[1]), __uint_as_float(r2[0]));
            }
            if constexpr (SUM) {
                const f32x4 tb = mfma16(*(const half8*)&ss[w][(l & 7u) * 32 + 8 * c], *(const half8*)&um[w][8 * l], z4);
#pragma unroll
                for (int e = 0; e < 4; e++) t[e] = __builtin_fmaf(32.0f, tb[e], t[e]);
                own();
            }
            if (c < 2)
#pragma unroll
                for (int e = 0; e < 4; e++) ps[u - u0][4 * c + e][l] = t[e];
        }
    };
    // The units' sums in order, split by split (k_matmul_mm's accumulation).
    const uint32_t i = tid >> 4, r = r0 + (tid & 15);
    const bool folds = tid < 128 && i < ni && r < p.rows;
    float acc = 0.0f, tot = 0.0f;
    uint32_t kz = 0, kend = p.units / p.ks;
    auto fold = [&](uint32_t u0, uint32_t ue) {
        if (!LONG && p.ks == 1) {
            for (uint32_t u = 0; u < ue; u++) tot = __builtin_fmaf(isc[u][i], ps[u][i][tid & 15], tot);
            return;
        }
        for (uint32_t u = u0; u < ue; u++) {
            acc = __builtin_fmaf(isc[u - u0][i], ps[u - u0][i][tid & 15], acc);
            if (u + 1 < kend) continue;
            tot = kz == 0 ? acc : tot + acc;
            acc = 0.0f;
            kz++;
            kend = (kz + 1) * p.units / p.ks;
        }
    };
    if constexpr (LONG) {
        for (uint32_t u0 = 0; u0 < p.units; u0 += WV_UNITS) {
            const uint32_t ue = min(u0 + WV_UNITS, p.units);
            stretch(u0, ue);
            __syncthreads();
            if (folds) fold(u0, ue);
            __syncthreads();  // the next stretch's sums take their place
        }
        if (!folds) return;
    } else {
        stretch(0, p.units);
        __syncthreads();
        if (!folds) return;
        fold(0, p.units);
    }
    p.out[(size_t)(i0 + i) * p.rows + r] = tot;
}

// FULL: cols is a multiple of 256, so a unit is four whole steps of straight-line code.
template <uint32_t TY, int TM, int TN, int WM, bool FULL>
__global__ __launch_bounds__(TL_THREADS, 2) void k_matmul_tile(const TLParams p) {
    constexpr int WN = 8 / WM, MT = 16 * TM * WM;
    static_assert(16 * TN * WN == TL_NT, "eight waves cover the weight rows");
    constexpr bool SUM = mm_sum<TY>(), KQ = tl_kq<TY>(), UT = KQ || TY == G_F16;
    constexpr int XL = MT * 16 / TL_THREADS;  // 16-byte pieces of x a thread moves a step
    static_assert(XL >= 1 && MT * 16 % TL_THREADS == 0 && 4 * MT <= TL_THREADS, "a step's x divides over the threads");
    // One LDS object a stage: the compiler then waits only for the stage it reads.
    __shared__ __attribute__((aligned(16))) uint8_t xl0[MT * 256], xl1[MT * 256], wl0[TL_NT * 128], wl1[TL_NT * 128];
    __shared__ __attribute__((aligned(16))) float is[2][MT];
    __shared__ float sa[2][UT ? 1 : (TY == G_Q6K ? 4 : 2) * TL_NT];
    __shared__ __attribute__((aligned(16))) float uf[2][KQ ? 2 * TL_NT : 1];
    __shared__ __attribute__((aligned(16))) f16 um[2][SUM ? 8 * (KQ ? 2 : 1) * TL_NT : 1];
    __shared__ __attribute__((aligned(16))) f16 us[2][SUM ? 32 * MT : 1];
    __shared__ uint32_t last;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t c = lane >> 4, l = lane & 15;
    // Workgroups 8 apart share an XCD: consecutive ones there take the input tiles of one
    // stretch of weight rows, so that its packed bytes come from the XCD's L2 after the first.
    const uint32_t xcd = blockIdx.x % 8, tile = xcd * (gridDim.x / 8) + min(xcd, gridDim.x % 8) + blockIdx.x / 8;
    const uint32_t wx = tile / p.nyt, wy = tile % p.nyt;
    const uint32_t r0 = wx * TL_NT, i0 = wy * MT;
    const uint32_t tr = tid >> 2, qd = tid & 3;  // the weight row and quarter this thread unpacks
    const uint8_t* wrow = p.w + (size_t)min(r0 + tr, p.rows - 1) * p.row_bytes;
    const uint32_t wm = wv / WN, wn = wv % WN;   // the wave's tiles: inputs 16 TM wm .., rows 16 TN wn ..
    const f32x4 z4 = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const uint32_t kz0 = p.par ? blockIdx.z : 0, kz1 = p.par ? blockIdx.z + 1 : p.ks;
    const uint32_t nsteps = (p.groups + 1) / 2;
    // LDS offsets of the lane's operands: piece 4 g + c of row l of a tile; x rows are 16
    // pieces swizzled by the row, weight rows 8 pieces swizzled by the row pair.
    const uint32_t xa = (16 * TM * wm + l) * 256, wa = (16 * TN * wn + l) * 128, wsw = (l >> 1) & 7u;
    uint32_t pk[2][TLP<TY>];  // packed weights of the next step and the one after
    uint32_t hd[TLH<TY>];     // the next unit's header
    MMUnit mu;
    u32x4 sr = u32x4{};
    float ir = 0.0f;
    // A step's x straight into its LDS stage, 1 KB (four rows) a wave and load; lane i fetches
    // the piece that belongs in its 16 bytes.
    auto fetch_x = [&](uint32_t s, uint8_t* dst) {
#pragma unroll
        for (int i = 0; i < XL; i++) {
            const uint32_t blk = wv * XL + i, row = 4 * blk + c;
            const uint8_t* base = (const uint8_t*)p.xp + ((size_t)s * p.npad + i0) * 256;  // uniform
            const uint32_t off = row * 256 + 16 * (l ^ (row & 15u));
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(base + off),
                                             (__attribute__((address_space(3))) void*)(dst + blk * 1024), 16, 0, 0);
        }
    };
    auto fetch_unit = [&](uint32_t u) {
        const size_t at = (size_t)u * p.npad + i0;
        tl_head<TY>(wrow, u, hd);
        ir = p.ip[at + min(tid, (uint32_t)MT - 1u)];
        if constexpr (SUM) sr = *(const u32x4*)(p.sp + at * 32 + 8 * min(tid, 4u * MT - 1u));
    };
    auto stash = [&](const uint32_t (&pw)[TLP<TY>], uint32_t s, uint32_t cc) {
        const uint32_t ub = (s >> 2) & 1;
        tl_stash<TY, FULL>(pw, hd, mu, s, cc, tr, qd, p.groups, cc & 1 ? wl1 : wl0, sa[cc & 1], uf[ub], um[ub]);
        if (cc == 0) {
            if (tid < (uint32_t)MT) is[ub][tid] = ir;
            if constexpr (SUM)
                if (tid < 4u * MT) *(u32x4*)(us[ub] + 8 * (tid ^ ((tid >> 4) & 3u))) = sr;
        }
    };
    f32x4 tot[TM][TN];
    for (uint32_t kz = kz0; kz < kz1; kz++) {
        const uint32_t ua = kz * p.units / p.ks, ue = (kz + 1) * p.units / p.ks;
        const uint32_t s1 = min(4 * ue, nsteps);
        // t and to: hi and lo (Q6K: both in t)
        f32x4 ac[TM][TN], t[TM][TN], to[TY == G_Q6K ? 1 : TM][TY == G_Q6K ? 1 : TN];
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) ac[i][j] = z4;
        if (kz != kz0) __syncthreads();  // the previous split's last step is read
        fetch_unit(ua);
        tl_load<TY>(wrow, 4 * ua, qd, p.groups, pk[0]);
        fetch_x(4 * ua, xl0);
        tl_load<TY>(wrow, min(4 * ua + 1, s1 - 1), qd, p.groups, pk[1]);
        stash(pk[0], 4 * ua, 0);
        __syncthreads();
        for (uint32_t u = ua; u < ue; u++) {
#pragma unroll
            for (uint32_t cc = 0; cc < 4; cc++) {
                const uint32_t s = 4 * u + cc;
                if (!FULL && s >= s1) break;
                // Step s + 1's x into the other stage, its packed weights (loaded a step ago)
                // unpacked beside this step's MFMAs, step s + 2's packed weights on their way.
                // (FULL: past the range's end its last step again into the stage no one reads any
                // more, so that no branch splits the unit: across one the compiler gathers every
                // step's FMAs at the unit's end and spills.)
                const uint8_t *xb = (cc & 1 ? xl1 : xl0) + xa, *wb = (cc & 1 ? wl1 : wl0) + wa;
                // The first operand before the new loads go out: the compiler waits for every load in
                // flight at a stage's first read, which then are only those of a step ago.
                const half8 xf = *(const half8*)(xb + 16 * (c ^ l));
                __builtin_amdgcn_sched_barrier(0);
                const bool more = FULL || s + 1 < s1;
                const uint32_t sn = min(s + 1, s1 - 1);
                if (more) {
                    if (cc == 2) fetch_unit(min(u + 1, ue - 1));
                    fetch_x(sn, cc & 1 ? xl0 : xl1);
                    __builtin_amdgcn_sched_barrier(0);
                    tl_load<TY>(wrow, min(s + 2, s1 - 1), qd, p.groups, pk[cc & 1]);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (uint32_t g = 0; g < 2; g++) {
                    if (!FULL && 2 * s + g >= p.groups) break;
                    half8 b[TN];
                    float a0[TN], a1[TN];
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        b[j] = *(const half8*)(wb + 2048 * j + 16 * ((4 * g + c) ^ wsw));
                        const uint32_t r = 16 * (TN * wn + j) + l;
                        if constexpr (TY == G_Q6K) {
                            a0[j] = sa[cc & 1][(2 * g) * TL_NT + r];
                            a1[j] = sa[cc & 1][(2 * g + 1) * TL_NT + r];
                        } else if constexpr (!UT) {
                            a0[j] = sa[cc & 1][g * TL_NT + r];
                        }
                    }
#pragma unroll
                    for (int i = 0; i < TM; i++) {
                        const uint32_t p0 = TY == G_Q6K ? 8 * g + c : 4 * g + c, p1 = TY == G_Q6K ? p0 + 4 : p0 + 8;
                        const half8 x0 = g == 0 && i == 0 ? xf : *(const half8*)(xb + 4096 * i + 16 * (p0 ^ l));
                        const half8 x1 = *(const half8*)(xb + 4096 * i + 16 * (p1 ^ l));
#pragma unroll
                        for (int j = 0; j < TN; j++) {
                            if constexpr (UT) {
                                t[i][j] = mfma16(x0, b[j], cc == 0 && g == 0 ? z4 : t[i][j]);
                                to[i][j] = mfma16(x1, b[j], cc == 0 && g == 0 ? z4 : to[i][j]);
                            } else if constexpr (TY == G_Q6K) {
                                const f32x4 h0 = mfma16(x0, __builtin_shufflevector(b[j], b[j], 0, 1, 2, 3, 0, 1, 2, 3), z4);
                                const f32x4 h1 = mfma16(x1, __builtin_shufflevector(b[j], b[j], 4, 5, 6, 7, 4, 5, 6, 7), z4);
#pragma unroll
                                for (int e = 0; e < 4; e++)
                                    t[i][j][e] = __builtin_fmaf(a1[j], h1[e], __builtin_fmaf(a0[j], h0[e], cc == 0 && g == 0 ? 0.0f : t[i][j][e]));
                            } else {
                                const f32x4 h = mfma16(x0, b[j], z4), o = mfma16(x1, b[j], z4);
#pragma unroll
                                for (int e = 0; e < 4; e++) {
                                    t[i][j][e] = __builtin_fmaf(a0[j], h[e], cc == 0 && g == 0 ? 0.0f : t[i][j][e]);
                                    to[i][j][e] = __builtin_fmaf(a0[j], o[e], cc == 0 && g == 0 ? 0.0f : to[i][j][e]);
                                }
                            }
                        }
                        // The FMAs stay here: the compiler otherwise sinks a unit's to its end, every
                        // MFMA's result kept until then, and spills.
                        if constexpr (!UT)
#pragma unroll
                            for (int j = 0; j < TN; j++) {
                                asm volatile("" : "+v"(t[i][j]));
                                if constexpr (TY != G_Q6K) asm volatile("" : "+v"(to[i][j]));
                            }
                    }
                }
                if (cc == 3 || (!FULL && s + 1 == s1)) {  // the unit's end
                    const uint32_t ub = u & 1;
                    float dl[TN], bl[TN];
                    half8 mv[TN];
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        const uint32_t r = 16 * (TN * wn + j) + l;
                        dl[j] = 1.0f;
                        bl[j] = 32.0f;
                        if constexpr (KQ) {
                            const float2 f = *(const float2*)(uf[ub] + 2 * r);
                            dl[j] = f.x;
                            bl[j] = f.y;
                        }
                        if constexpr (SUM) mv[j] = *(const half8*)(um[ub] + 8 * (KQ && c != 0 ? r + TL_NT : r));
                    }
#pragma unroll
                    for (int i = 0; i < TM; i++) {
                        const f32x4 i4 = *(const f32x4*)&is[ub][16 * (TM * wm + i) + 4 * c];
                        half8 sv;
                        if constexpr (SUM) {
                            const uint32_t e = 4 * (16 * (TM * wm + i) + l) + c;
                            sv = *(const half8*)(us[ub] + 8 * (e ^ ((e >> 4) & 3u)));
                        }
#pragma unroll
                        for (int j = 0; j < TN; j++) {
                            f32x4 v = t[i][j];
                            if constexpr (TY != G_Q6K)
#pragma unroll
                                for (int e = 0; e < 4; e++) v[e] = __builtin_fmaf(MM_LO_INV, to[i][j][e], v[e]);
                            if constexpr (KQ) v *= dl[j];
                            if constexpr (SUM) {
                                const f32x4 tb = mfma16(sv, mv[j], z4);
#pragma unroll
                                for (int e = 0; e < 4; e++) v[e] = __builtin_fmaf(bl[j], tb[e], v[e]);
                            }
#pragma unroll
                            for (int e = 0; e < 4; e++) ac[i][j][e] = __builtin_fmaf(i4[e], v[e], ac[i][j][e]);
                        }
                    }
                }
                if (more) stash(pk[(cc + 1) & 1], sn, (cc + 1) & 3);
                // The next step's x has landed (of the loads in flight only the last weight loads,
                // TLN or more, may be left) and its LDS writes are done. (__syncthreads would wait
                // for every load.)
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(TLN<TY>) : "memory");
            }
        }
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) tot[i][j][e] = kz == kz0 ? ac[i][j][e] : tot[i][j][e] + ac[i][j][e];
    }
    // Element e of tile (i, j) in lane (c, l): input 4c + e, weight row l.
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t in = i0 + 16 * (TM * wm + i) + 4 * c + e;
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const uint32_t r = r0 + 16 * (TN * wn + j) + l;
                if (r >= p.rows) continue;
                if (p.par)
                    __hip_atomic_store(&p.part[((size_t)blockIdx.z * p.npad + in) * p.rows + r], tot[i][j][e],
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                else if (in < p.n)
                    p.out[(size_t)in * p.rows + r] = tot[i][j][e];
            }
        }
    if (!p.par) return;
    // Parallel splits, as k_matmul_mm's: the tile's last workgroup adds the partials in order.
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) {
        const uint32_t old = __hip_atomic_fetch_add(&p.cnt[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = old == p.ks - 1;
    }
    __syncthreads();
    if (!last) return;
    const size_t stride = (size_t)p.npad * p.rows;
    const uint32_t rr = r0 + tid % TL_NT;
    constexpr uint32_t IP = TL_THREADS / TL_NT;  // inputs a pass of the workgroup
    for (uint32_t q = 0; q < (uint32_t)MT; q += 2 * IP) {
        float sum[2] = {0.0f, 0.0f};
        for (uint32_t k0 = 0; k0 < p.ks; k0 += 8) {
            float v[2][8];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const float* src = p.part + (size_t)(i0 + q + IP * h + tid / TL_NT) * p.rows + min(rr, p.rows - 1);
#pragma unroll
                for (int t = 0; t < 8; t++)
                    v[h][t] = k0 + t < p.ks ? __hip_atomic_load(src + (k0 + t) * stride, __ATOMIC_RELAXED,
                                                                 __HIP_MEMORY_SCOPE_AGENT)
                                            : 0.0f;
            }
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int t = 0; t < 8; t++)
                    if (k0 + t < p.ks) sum[h] = k0 + t == 0 ? v[h][t] : sum[h] + v[h][t];
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t in = i0 + q + IP * h + tid / TL_NT;
            if (in < p.n && rr < p.rows) p.out[(size_t)in * p.rows + rr] = sum[h];
        }
    }
    if (tid == 0) __hip_atomic_store(&p.cnt[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Rows a workgroup of the format takes.
static uint32_t mm_rows(uint32_t type) {
    return type == G_F16 ? 16 * MM_W<G_F16> : 16 * MM_W<G_Q4K>;
}
// K splits of a product: about two workgroups a CU from the rows alone (never from n), each
// split at most MM_K units.
static uint32_t mm_ks(uint32_t type, uint32_t rows, uint32_t cols) {
    const uint32_t rt = (rows + mm_rows(type) - 1) / mm_rows(type), units = (cols + 255) / 256;
    const uint32_t kmax = type == G_F16 ? MM_K<G_F16> : MM_K<G_Q4K>;
    if (cols % 256 != 0 && units <= 16) return 1;  // (no k_matmul_mm form: short ranges stay whole)
    uint32_t ks = max(512u / rt, 1u);
    ks = max(ks, (units + kmax - 1) / kmax);
    ks = min(ks, units);
    return max(ks, 1u);
}
static bool mm_par(uint32_t type, uint32_t rows, uint32_t cols, uint32_t n) {
    const uint32_t rt = (rows + mm_rows(type) - 1) / mm_rows(type), nt = (n + 7) / 8;
    return mm_ks(type, rows, cols) > 1 && (uint64_t)rt * nt <= MM_PAR;
}

static bool mm_types(uint32_t type) {
    switch (type) {
        case G_F16: case G_Q8_0: case G_Q4_0: case G_Q4_1: case G_Q5_0: case G_Q5_1: case G_Q4K: case G_Q5K:
        case G_Q6K: return true;
        default: return false;
    }
}

static bool matmul_uses_mm(uint32_t type, uint32_t cols, uint32_t n) {
    return mm_types(type) && n >= MM_MIN && cols % 256 == 0;
}

// Bytes of prepared x a launch takes at most, and its input rows (k_mm_prep's grid.y is a quarter of
// them, of 65535); longer batches go in slabs of input rows.
constexpr size_t TL_SLAB_BYTES = (size_t)256 << 20, TL_SLAB_ROWS = 4 * 65535;

static bool matmul_uses_units(uint32_t type, uint32_t cols, uint32_t n) {
    return mm_types(type) && cols % 256 != 0 && n >= MM_MIN;
}
struct TilePlan {
    uint32_t mt, slab, npad, units, groups, ks, nxt, nyt, par;  // npad, nyt, par: of a whole slab
    size_t xp_bytes, ip_bytes, sp_bytes, part_bytes;
};
static TilePlan tile_plan(uint32_t type, uint32_t rows, uint32_t cols, uint32_t n) {
    TilePlan t{};
    t.units = (cols + 255) / 256;
    t.groups = cols / 32;
    t.nxt = (rows + TL_NT - 1) / TL_NT;
    const size_t row_bytes = (size_t)(t.groups + 1) / 2 * 256;
    t.slab = (uint32_t)std::max<size_t>(std::min(TL_SLAB_BYTES / row_bytes, TL_SLAB_ROWS) / 128 * 128, 128);
    const uint32_t m = min(n, t.slab);
    // Input rows a workgroup: 128 where that still gives every CU one.
    t.mt = m <= 32 ? 32 : (m > 64 && (uint64_t)t.nxt * ((m + 127) / 128) >= 256) ? 128 : 64;
    t.npad = (m + t.mt - 1) / t.mt * t.mt;
    t.nyt = t.npad / t.mt;
    t.ks = mm_ks(type, rows, cols);
    // K splits in parallel where the tiles alone would leave half the CUs without work, or, 32 inputs
    // a workgroup, some of them (18944 x 3584, 148 tiles, at 17 rows: Q4K 39 -> 31 us, Q8_0 59 -> 45).
    t.par = t.ks > 1 && (uint64_t)t.nxt * t.nyt <= (t.mt == 32 ? 255 : 128);
    t.xp_bytes = (size_t)t.npad * row_bytes;
    t.ip_bytes = ((size_t)t.units * t.npad * sizeof(float) + 255) / 256 * 256;
    t.sp_bytes = (size_t)t.units * t.npad * 64;
    t.part_bytes = t.par ? (size_t)t.ks * t.npad * rows * sizeof(float) : 0;
    return t;
}

// Which kernel takes a batch of the matrix-core formats; all give an input row the same bits. The
// tile kernel's work goes by its padded input rows, k_matmul_mm's and k_matmul_units' by eights, so
// over them it takes batches of 17 rows with enough multiply-adds, by what the unpacking it saves costs,
// that fill its tiles enough (us there / here):
//   F16 1024 x 4096 at 33 rows (0.14 G) 28 / 24;
//   Q8_0, Q6K 4096 x 4096 at 48 rows (0.8 G) 36 / 33 and 38 / 34, at 40 30 / 33 and 33 / 34;
//   the others 3584 x 3584 at 80 rows (1.0 G) Q4K 41 / 42, at 96 48 / 42; 33 rows in a tile of 64
//   4096 x 14336 Q4K 44 / 48, 8192 x 8192 45 / 42, but not for a few tiles more than CUs (18944 x 3584 at
//   65 rows, 296 of them, 89 / 97);
//   Q4_0, Q5_0 (cheap to unpack) 4096 x 14336 at 64 rows Q4_0 60 / 54, at 80 76 / 90, at 112 105 / 90;
//   off a multiple of 256 4864 x 896 at 40 rows (0.17 G) Q8_0 15 / 19, at 48 18 / 19, at 56 21 / 19.
constexpr uint32_t TL_MIN = 17;
constexpr uint64_t TL_MACS_F16 = 100000000, TL_MACS_8 = 760000000, TL_MACS = 900000000, TL_MACS_4 = 1200000000,
                   TL_MACS_4_ANY = 5000000000, TL_MACS_RAGGED = 200000000;

bool matmul_uses_tile(uint32_t type, uint32_t rows, uint32_t cols, uint32_t n) {
    const uint64_t macs = (uint64_t)rows * cols * n;
    if (!mm_types(type)) return false;
    if (cols % 256 != 0) return n >= MM_MIN && ((cols + 255) / 256 > WV_UNITS || (n >= TL_MIN && macs >= TL_MACS_RAGGED));
    if (n < TL_MIN) return false;
    const TilePlan t = tile_plan(type, rows, cols, n);
    const uint64_t eights = 100ull * ((min(n, t.slab) + 7) / 8 * 8);  // of npad, in percent
    const uint32_t tiles = t.nxt * t.nyt;
    switch (type) {
        case G_F16: return macs >= TL_MACS_F16;
        case G_Q4_0: case G_Q5_0: return macs >= TL_MACS_4 && (eights >= 80ull * t.npad || macs >= TL_MACS_4_ANY);
        default:
            return macs >= (type == G_Q8_0 || type == G_Q6K ? TL_MACS_8 : TL_MACS) &&
                   (eights >= 65ull * t.npad || (rows >= 8192 && (tiles <= 256 || tiles > 384)));
    }
}

size_t matmul_scratch_bytes(uint32_t type, uint32_t rows, uint32_t cols, uint32_t n, bool tile) {
    if (tile) {
        const TilePlan t = tile_plan(type, rows, cols, n);
        return t.xp_bytes + t.ip_bytes + t.sp_bytes + t.part_bytes;
    }
    if (!matmul_uses_mm(type, cols, n) || !mm_par(type, rows, cols, n)) return 0;
    return (size_t)mm_ks(type, rows, cols) * ((n + 15) / 16 * 16) * rows * sizeof(float);
}

template <uint32_t TY>
static hipError_t matmul_mm_go(const MatmulParams& mp, void* scratch, uint32_t* counters, hipStream_t s) {
    const uint32_t ks = mm_ks(TY, mp.rows, mp.cols), rt = (mp.rows + 16 * MM_W<TY> - 1) / (16 * MM_W<TY>);
    const bool par = scratch && counters && mm_par(TY, mp.rows, mp.cols, mp.n);  // (else in turn: the same bits)
    const MMParams q{mp.w, mp.x, mp.out, (float*)scratch, counters, mp.rows, mp.cols, mp.n, (mp.n + 15) / 16 * 16,
                     mp.row_bytes, mp.cols / 256, ks, par ? 1u : 0u};
    // Sixteen inputs a workgroup (9 to 16 rows) halve the unpacking but leave one workgroup a CU, so
    // they pay where a split holds several units, the sooner the dearer the unpacking; us at 9 / 16
    // rows with eight and with sixteen: 14336 x 4096 (four units) Q6K 32.1 / 33.3 and 26.6 / 28.3, Q8_0
    // 28.4 / 29.1 and 25.6 / 26.8, Q5K 25.4 / 26.5 and 22.9 / 24.8; 4096 x 4096 (one) 15.7 / 15.9 and
    // 15.8 / 16.4, 15.0 / 15.2 and 15.7 / 16.4, 14.1 / 14.8 and 14.8 / 15.8. Q4K only where the
    // workgroups also go around the CUs four times: 28672 x 8192 71 / 75 and 65 / 71, 4096 x 14336 21.4 /
    // 21.9 and 21.4 / 23.2. Q4_0, Q4_1 and Q5_1 lost or gained nothing. (F16's x of 16 inputs would
    // take most of the LDS.)
    constexpr uint32_t MIN_UNITS = TY == G_Q6K ? 2 : TY == G_Q8_0 || TY == G_Q5_0 || TY == G_Q4K || TY == G_Q5K ? 3 : 0;
    if constexpr (MIN_UNITS > 0) {
        if (mp.n > 8 && mp.n <= 16 && q.units >= MIN_UNITS * ks && (TY != G_Q4K || rt * ks >= 1024)) {
            const dim3 grid(rt, (mp.n + 15) / 16, par ? ks : 1);
            hipLaunchKernelGGL((k_matmul_mm<TY, 16>), grid, dim3(64 * MM_W<TY>), 0, s, q);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((k_matmul_mm<TY, 8>), dim3(rt, (mp.n + 7) / 8, par ? ks : 1), dim3(64 * MM_W<TY>), 0, s, q);
    return hipGetLastError();
}

static bool matmul_uses_row(uint32_t type, uint32_t cols, uint32_t n) {
    return n == 1 && mm_types(type) && type != G_F16 && cols % 256 == 0 && cols / 256 <= ROW_UNITS;
}
template <uint32_t TY>
static hipError_t matmul_row_go(const MatmulParams& mp, hipStream_t s) {
    const uint32_t units = mp.cols / 256;
    const MMParams q{mp.w, mp.x, mp.out, nullptr, nullptr, mp.rows, mp.cols, 1, 1, mp.row_bytes, units, 1, 0};
    const size_t lds = (size_t)units * (16 * sizeof(double) + sizeof(float));
    const dim3 grid((mp.rows + 15) / 16);
    // Sixteen waves a workgroup where there is at most one a CU, eight where there are more.
    // (with f32 sums at the end) 4096 x 14336 at sixteen and eight: Q4K 13.1 and 14.3 us, Q6K 18.7
    // and 20.1; 14336 x 4096: 15.5 and 11.9, 22.6 and 18.9; 8192 x 28672: 40.9 and 39.0. Up to sixteen
    // units a wave has one: 3584 x 3584 Q4K 6.3 -> 5.8 us without the second load and the loop.
    if (mp.rows > 4096)
        hipLaunchKernelGGL((k_matmul_row<TY, 8, false>), grid, dim3(512), lds, s, q);
    else if (units > 16)
        hipLaunchKernelGGL((k_matmul_row<TY, 16, false>), grid, dim3(1024), lds, s, q);
    else
        hipLaunchKernelGGL((k_matmul_row<TY, 16, true>), grid, dim3(1024), lds, s, q);
    return hipGetLastError();
}

template <uint32_t TY>
static hipError_t matmul_units_go(const MatmulParams& mp, hipStream_t s) {
    const uint32_t units = (mp.cols + 255) / 256;
    const TLParams q{mp.w, nullptr, nullptr, nullptr, mp.out, nullptr, nullptr, mp.rows, mp.n, 0, mp.row_bytes,
                     units, mp.cols / 32, mm_ks(TY, mp.rows, mp.cols), 0, 0};
    const dim3 grid((mp.rows + 15) / 16, (mp.n + 7) / 8);
    if (units <= 4)
        hipLaunchKernelGGL((k_matmul_units<TY, 4, false>), grid, dim3(256), 0, s, q, mp.x, mp.cols);
    else if (units <= WV_UNITS)
        hipLaunchKernelGGL((k_matmul_units<TY, 8, false>), grid, dim3(512), 0, s, q, mp.x, mp.cols);
    else
        hipLaunchKernelGGL((k_matmul_units<TY, 8, true>), grid, dim3(512), 0, s, q, mp.x, mp.cols);
    return hipGetLastError();
}

template <uint32_t TY>
static hipError_t matmul_tile_go(const MatmulParams& mp, void* scratch, uint32_t* counters, hipStream_t s) {
    const TilePlan t = tile_plan(TY, mp.rows, mp.cols, mp.n);
    if (!scratch || !counters) return hipErrorInvalidValue;
    f16* xp = (f16*)scratch;
    float* ip = (float*)((char*)scratch + t.xp_bytes);
    f16* sp = (f16*)((char*)ip + t.ip_bytes);
    float* part = (float*)((char*)sp + t.sp_bytes);
    for (uint32_t n0 = 0; n0 < mp.n; n0 += t.slab) {
        const uint32_t m = min(mp.n - n0, t.slab), nyt = (m + t.mt - 1) / t.mt, npad = nyt * t.mt;
        hipLaunchKernelGGL((k_mm_prep<tl_order<TY>(), tl_kq<TY>() ? 2 : mm_sum<TY>() ? 1 : 0>), dim3(t.units, npad / 4), dim3(256), 0, s,
                           mp.x + (size_t)n0 * mp.cols, xp, ip, sp, m, mp.cols, npad, (t.groups + 1) / 2);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        const TLParams q{mp.w, xp, ip, sp, mp.out + (size_t)n0 * mp.rows, part, counters, mp.rows, m, npad, mp.row_bytes,
                         t.units, t.groups, t.ks, t.par, nyt};
        const dim3 grid(t.nxt * nyt, 1, t.par ? t.ks : 1);
        auto go = [&](auto full) {
            constexpr bool FULL = decltype(full)::value;
            if (t.mt == 128)
                hipLaunchKernelGGL((k_matmul_tile<TY, 2, 4, 4, FULL>), grid, dim3(TL_THREADS), 0, s, q);
            else if (t.mt == 64)
                hipLaunchKernelGGL((k_matmul_tile<TY, 2, 2, 2, FULL>), grid, dim3(TL_THREADS), 0, s, q);
            else
                hipLaunchKernelGGL((k_matmul_tile<TY, 2, 1, 1, FULL>), grid, dim3(TL_THREADS), 0, s, q);
        };
        if (mp.cols % 256 == 0) {
            go(std::true_type{});
        } else if constexpr (!tl_kq<TY>() && TY != G_Q6K) {
            go(std::false_type{});
        }
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <uint32_t TY, int NBT, int R>
static void matmul_go(const MatmulParams& mp, hipStream_t s) {
    const uint32_t per_wg = MM_WAVES * R;
    const dim3 grid((mp.rows + per_wg - 1) / per_wg, (mp.n + NBT - 1) / NBT);
    const size_t lds = (size_t)min(mp.n, (uint32_t)NBT) * TILE_GROUPS * XS * sizeof(float);
    hipLaunchKernelGGL((k_matmul<TY, NBT, R>), grid, dim3(64 * MM_WAVES), lds, s, mp);
}

// One input row in the vector-unit pass (the plain types, and cols off a multiple of 256 or
// beyond ROW_UNITS units): eight rows a wave when a group packs into at most 12 dwords and
// the matrix still gives 256+ workgroups (measured: the 14336 x 4096 Q4K product 21.3 ->
// 14.2 µs), else four. Batches: four rows a wave, eight input rows a pass.
template <uint32_t TY>
static hipError_t matmul_t(const MatmulParams& mp, bool tile, void* scratch, uint32_t* counters, hipStream_t s) {
    if constexpr (mm_type<TY>()) {
        if (tile) return matmul_tile_go<TY>(mp, scratch, counters, s);
        if constexpr (!tl_kq<TY>() && TY != G_Q6K)
            if (matmul_uses_units(TY, mp.cols, mp.n)) return matmul_units_go<TY>(mp, s);
        if (matmul_uses_mm(TY, mp.cols, mp.n)) return matmul_mm_go<TY>(mp, scratch, counters, s);
        if constexpr (MM_LDSP<TY>)
            if (matmul_uses_row(TY, mp.cols, mp.n)) return matmul_row_go<TY>(mp, s);
    }
    if (mp.n == 1) {
        if (PK<TY> <= 12 && mp.rows >= 256u * MM_WAVES * 8)
            matmul_go<TY, 1, (PK<TY> <= 12 ? 8 : 4)>(mp, s);
        else
            matmul_go<TY, 1, 4>(mp, s);
    } else {
        matmul_go<TY, NB, 4>(mp, s);
    }
    return hipGetLastError();
}

hipError_t matmul_launch(const void* w, uint32_t type, const float* x, float* out, uint32_t rows, uint32_t cols,
                         uint32_t n, uint32_t row_bytes, bool tile, void* scratch, uint32_t* counters, hipStream_t s) {
    const MatmulParams mp{(const uint8_t*)w, x, out, rows, cols, n, row_bytes};
    switch (type) {
        case G_F32: return matmul_t<G_F32>(mp, tile, scratch, counters, s);
        case G_F16: return matmul_t<G_F16>(mp, tile, scratch, counters, s);
        case G_BF16: return matmul_t<G_BF16>(mp, tile, scratch, counters, s);
        case G_Q4_0: return matmul_t<G_Q4_0>(mp, tile, scratch, counters, s);
        case G_Q4_1: return matmul_t<G_Q4_1>(mp, tile, scratch, counters, s);
        case G_Q5_0: return matmul_t<G_Q5_0>(mp, tile, scratch, counters, s);
        case G_Q5_1: return matmul_t<G_Q5_1>(mp, tile, scratch, counters, s);
        case G_Q8_0: return matmul_t<G_Q8_0>(mp, tile, scratch, counters, s);
        case G_Q4K: return matmul_t<G_Q4K>(mp, tile, scratch, counters, s);
        case G_Q5K: return matmul_t<G_Q5K>(mp, tile, scratch, counters, s);
        case G_Q6K: return matmul_t<G_Q6K>(mp, tile, scratch, counters, s);
        default: return hipErrorInvalidValue;
    }
}

// RMSNorm, one workgroup a row: the sum of squares over the workgroup's threads (4 values
// each step, a fixed tree), scale = 1 / sqrt(mean + eps), out = x * scale * w.
constexpr int NORM_THREADS = 256;

// vec: cols % 4 == 0 and every pointer 16-byte aligned (float4 accesses).
__global__ __launch_bounds__(NORM_THREADS) void k_rms_norm(const float* __restrict__ x, const float* __restrict__ w,
                                                           float* __restrict__ out, uint32_t cols, float eps,
                                                           bool vec) {
    __shared__ float part[NORM_THREADS / 64];
    const float* xr = x + (size_t)blockIdx.x * cols;
    float* orow = out + (size_t)blockIdx.x * cols;
    const uint32_t t = threadIdx.x;
    float s = 0.0f;
    if (vec) {
        for (uint32_t c = 4 * t; c < cols; c += 4 * NORM_THREADS) {
            const float4 v = *(const float4*)(xr + c);
            s += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
        }
    } else {
        for (uint32_t c = t; c < cols; c += NORM_THREADS) s += xr[c] * xr[c];
    }
    s = wave_sum(s);
    if ((t & 63) == 0) part[t >> 6] = s;
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int i = 0; i < NORM_THREADS / 64; i++) tot += part[i];
    const float scale = 1.0f / __builtin_sqrtf(tot / (float)cols + eps);
    if (vec) {
        for (uint32_t c = 4 * t; c < cols; c += 4 * NORM_THREADS) {
            const float4 v = *(const float4*)(xr + c), g = *(const float4*)(w + c);
            *(float4*)(orow + c) = float4{v.x * scale * g.x, v.y * scale * g.y, v.z * scale * g.z, v.w * scale * g.w};
        }
    } else {
        for (uint32_t c = t; c < cols; c += NORM_THREADS) orow[c] = xr[c] * scale * w[c];
    }
}

hipError_t rms_norm_launch(const float* x, const float* w, float* out, uint32_t rows, uint32_t cols, float eps,
                           bool vec, hipStream_t s) {
    hipLaunchKernelGGL(k_rms_norm, dim3(rows), dim3(NORM_THREADS), 0, s, x, w, out, cols, eps, vec);
    return hipGetLastError();
}

// Elementwise ops, grid-stride. silu's e^-v is 2^(-v log2 e) on the hardware's exp2, as the
// reference kernels compute it (cuda.cu:66).

template <int OP>
__global__ __launch_bounds__(256) void k_elementwise(float* __restrict__ x, const float* __restrict__ y, uint64_t n,
                                                     uint32_t dim) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        if constexpr (OP == EW_BIAS) {
            x[i] += y[i % dim];
        } else if constexpr (OP == EW_SILU_MUL) {
            const float v = x[i];
            x[i] = v / (1.0f + __builtin_amdgcn_exp2f(-v * LOG2E)) * y[i];
        } else {
            x[i] += y[i];
        }
    }
}

hipError_t elementwise_launch(int op, float* x, const float* y, uint64_t n, uint32_t dim, hipStream_t s) {
    const uint64_t blocks64 = (n + 255) / 256;
    const uint32_t blocks = (uint32_t)(blocks64 < 8192 ? blocks64 : 8192);
    switch (op) {
        case EW_BIAS: hipLaunchKernelGGL(k_elementwise<EW_BIAS>, dim3(blocks), dim3(256), 0, s, x, y, n, dim); break;
        case EW_SILU_MUL:
            hipLaunchKernelGGL(k_elementwise<EW_SILU_MUL>, dim3(blocks), dim3(256), 0, s, x, y, n, dim);
            break;
        default: hipLaunchKernelGGL(k_elementwise<EW_ADD>, dim3(blocks), dim3(256), 0, s, x, y, n, dim); break;
    }
    return hipGetLastError();
}

}  // namespace bchip
