// Rotary position embedding, fused with the type conversion and the write into its destination
// (a query tensor for the attention call, or the new rows of the KV cache).
//
// Semantics: fusor-ml/fusor/src/composite/rope.rs:46-137 in f32, one rounding per operation as the
// reference's CPU path has (mul, mul, add are separate tensor ops there):
//   normal (rope / rope_normal_fused):       y[i]        = x[i] * cos[p][i]        + (-x[i + D/2]) * sin[p][i]
//                                            y[i + D/2]  = x[i + D/2] * cos[p][i]  +   x[i]        * sin[p][i]
//   interleaved (rope_interleaved / rope_fused): y[2i]   = x[2i] * cos[p][i] - x[2i+1] * sin[p][i]
//                                            y[2i+1]     = x[2i] * sin[p][i] + x[2i+1] * cos[p][i]
// with p = start_pos + row (RopeCache::forward, rope.rs:232-265) and cos/sin the [positions, D/2]
// f32 tables of fusor::RopeCache.  16-bit inputs are widened to f32 first and the result is rounded
// to nearest even, which is what kalosm-llama's cast -> rope -> cast does
// (models/kalosm-llama/src/raw/rope.rs:103-111).
//
// Optionally the row is RMS-normalised first (the q / k norm of Qwen3- and Gemma3-style blocks,
// models/kalosm-llama/src/raw/attention_layer.rs:229-235,251-257 -> RmsNorm::forward_generic_4d,
// fusor-ml/fusor/src/layers/rms_norm.rs:122-133 -> rms_norm_fused_cpu_impl,
// fusor-ml/fusor/src/composite/normalization.rs:351-407), again one rounding per operation and in the
// reference's order:
//   ss = fold(+, 0, x[i] * x[i]) left to right;  rms = sqrt(ss / D + eps);  n[i] = (x[i] / rms) * w[i] (+ bias[i])
// and n is rounded to the tensor's element type before the rotation, because the reference's norm returns a
// tensor of that type.
#include <stddef.h>

#include "common.h"
#include "device_utils.h"

namespace fhip {

__device__ __forceinline__ float load_as_f32(const void *p, int64_t idx, int dtype) {
    if (dtype == FHIP_F32) return ((const float *)p)[idx];
    if (dtype == FHIP_F16) return (float)((const half_t *)p)[idx];
    return to_float(((const bf16_t *)p)[idx]);
}
__device__ __forceinline__ void store_from_f32(void *p, int64_t idx, int dtype, float v) {
    if (dtype == FHIP_F32) ((float *)p)[idx] = v;
    else if (dtype == FHIP_F16) ((half_t *)p)[idx] = (half_t)v;
    else ((bf16_t *)p)[idx] = from_float<bf16_t>(v);
}

__device__ __forceinline__ float round_through(float v, int dtype) {
    if (dtype == FHIP_F16) return (float)(half_t)v;
    if (dtype == FHIP_BF16) return to_float(from_float<bf16_t>(v));
    return v;
}

// x and y in bf16, packed (to nearest even; NaN stays NaN, quiet)
__device__ __forceinline__ uint32_t bf16_pair(float x, float y) {
    uint32_t r;
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
    return r;
}

// ---- 16 bytes (f32) / 8 bytes (16-bit) at a time -------------------------------------------------
// The fast forms below need rows whose elements are consecutive and whose starts are aligned to four
// elements on both sides, and a head_dim that is a multiple of 8 (fill_row_job checks; `vec`).
typedef uint32_t uint2r_t __attribute__((ext_vector_type(2)));

// Four elements as they lie in memory, and widened: apart, so that a lane's loads are all on their way before it waits for
// the first.
template <int DTYPE>
struct Raw4 {
    uint2r_t w;
    __device__ __forceinline__ void load(const void *p, int64_t idx) { w = *(const uint2r_t *)((const uint16_t *)p + idx); }
    __device__ __forceinline__ float4_t widened() const {
        float4_t v;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if constexpr (DTYPE == FHIP_F16) v[e] = (float)__builtin_bit_cast(half_t, (uint16_t)(w[e >> 1] >> (16 * (e & 1))));
            else v[e] = __uint_as_float(e & 1 ? w[e >> 1] & 0xffff0000u : w[e >> 1] << 16);
        }
        return v;
    }
};
template <>
struct Raw4<FHIP_F32> {
    uint4_t w;
    __device__ __forceinline__ void load(const void *p, int64_t idx) { w = *(const uint4_t *)((const float *)p + idx); }
    __device__ __forceinline__ float4_t widened() const { return __builtin_bit_cast(float4_t, w); }
};
// four values in a 16-bit type, packed
template <int DTYPE>
__device__ __forceinline__ uint2r_t packed4(float4_t v) {
    if constexpr (DTYPE == FHIP_BF16) return uint2r_t{bf16_pair(v[0], v[1]), bf16_pair(v[2], v[3])};
    uint32_t bits[4];
#pragma unroll
    for (int e = 0; e < 4; e++) bits[e] = (uint32_t)__builtin_bit_cast(uint16_t, (half_t)v[e]);
    return uint2r_t{bits[0] | (bits[1] << 16), bits[2] | (bits[3] << 16)};
}
// four values rounded to an element type
template <int DTYPE>
__device__ __forceinline__ float4_t rounded4(float4_t v) {
    if constexpr (DTYPE == FHIP_F32) {
        return v;
    } else {
        Raw4<DTYPE> r;
        r.w = packed4<DTYPE>(v);
        return r.widened();
    }
}
__device__ __forceinline__ void store4_from_f32(void *p, int64_t idx, int dtype, float4_t v) {
    if (dtype == FHIP_F32) *(float4_t *)((float *)p + idx) = v;
    else *(uint2r_t *)((uint16_t *)p + idx) = dtype == FHIP_F16 ? packed4<FHIP_F16>(v) : packed4<FHIP_BF16>(v);
}

// element offsets of row t (a flat index over [B, heads, rows], or over [B, rows, heads]) in the source and the destination, and
// its position
__device__ __forceinline__ void row_bases(const RopeRows &a, int64_t t, bool heads_first, int64_t *sb, int64_t *db, uint32_t *r) {
    const int inner = heads_first ? 1 : 2;
    const uint32_t i = (uint32_t)(t % a.shape[inner]);
    t /= a.shape[inner];
    const uint32_t o = (uint32_t)(t % a.shape[3 - inner]);
    const int64_t h = heads_first ? i : o, b = t / a.shape[3 - inner];
    *r = heads_first ? o : i;
    *sb = b * a.ss[0] + h * a.ss[1] + *r * a.ss[2];
    *db = b * a.ds[0] + h * a.ds[1] + *r * a.ds[2];
}

// t / d for the divisor whose (mul, shift) the host worked out (fill_row_job): exact for t < 2^31
__device__ __forceinline__ uint32_t divided(uint32_t t, uint32_t mul, uint32_t shift) { return mul ? __umulhi(t, mul) >> shift : t; }
__device__ __forceinline__ void row_bases_small(const RopeRows &a, uint32_t t, bool heads_first, int64_t *sb, int64_t *db, uint32_t *r) {
    uint32_t b, h;
    if (heads_first) {
        const uint32_t br = divided(t, a.mul[1], a.shift[1]);
        b = divided(br, a.mul[0], a.shift[0]);
        h = t - br * a.shape[1];
        *r = br - b * a.shape[2];
    } else {
        const uint32_t bh = divided(t, a.mul[0], a.shift[0]);
        b = divided(bh, a.mul[1], a.shift[1]);
        h = bh - b * a.shape[1];
        *r = t - bh * a.shape[2];
    }
    *sb = b * a.ss[0] + h * a.ss[1] + *r * a.ss[2];
    *db = b * a.ds[0] + h * a.ds[1] + *r * a.ds[2];
}

// RopeRows::few of the wide normalised form: what its rows per block are divided by, and whether its blocks take the heads of a
// position together
constexpr int NORM_FEW = 7, NORM_HEADS_FIRST = 8;

// The workgroups of a launch that work on one job: `at` of `count`.
struct JobBlocks {
    uint32_t at, count;
};

// Rotation / conversion without the norm, four pairs (or four elements) per lane and step: every load and store is
// 16 bytes of f32 or 8 bytes of a 16-bit type, consecutive lanes take consecutive pieces of a row.
template <bool SMALL, int SRC>
__device__ __forceinline__ void rope_rows_vec_body(const RopeRows &a, JobBlocks jb) {
    const uint32_t D = a.shape[3], half = D / 2;
    const uint32_t upr = a.mode == 2 ? D / 4 : half / 4;  // steps per row
    const int64_t total = (int64_t)a.shape[0] * a.shape[1] * a.shape[2] * upr;
    for (int64_t idx = (int64_t)jb.at * 256 + threadIdx.x; idx < total; idx += (int64_t)jb.count * 256) {
        int64_t sb, db;
        uint32_t r, j;
        if constexpr (SMALL) {
            const uint32_t row = divided((uint32_t)idx, a.mul[2], a.shift[2]);
            j = (uint32_t)idx - row * upr;
            row_bases_small(a, row, false, &sb, &db, &r);
        } else {
            j = (uint32_t)(idx % upr);
            row_bases(a, idx / upr, false, &sb, &db, &r);
        }
        Raw4<SRC> p0, p1;
        if (a.mode == 2) {
            p0.load(a.src, sb + 4 * j);
            store4_from_f32(a.dst, db + 4 * j, a.dst_dtype, p0.widened());
            continue;
        }
        // the pieces of a step: (4j, half + 4j) or, interleaved, (8j, 8j + 4)
        const uint32_t d0 = a.mode == 0 ? 4 * j : 8 * j, d1 = a.mode == 0 ? half + 4 * j : 8 * j + 4;
        p0.load(a.src, sb + d0);
        p1.load(a.src, sb + d1);
        const float4_t c = *(const float4_t *)(a.cos + (a.pos0 + r) * half + 4 * j);
        const float4_t s = *(const float4_t *)(a.sin + (a.pos0 + r) * half + 4 * j);
        const float4_t xa = p0.widened(), xb = p1.widened();
        float4_t ya, yb;
        if (a.mode == 0) {  // pairs (4j + e, half + 4j + e)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                ya[e] = __fsub_rn(__fmul_rn(xa[e], c[e]), __fmul_rn(xb[e], s[e]));
                yb[e] = __fadd_rn(__fmul_rn(xb[e], c[e]), __fmul_rn(xa[e], s[e]));
            }
        } else {  // pairs (8j + 2e, 8j + 2e + 1)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float x0 = e < 2 ? xa[2 * e] : xb[2 * e - 4], x1 = e < 2 ? xa[2 * e + 1] : xb[2 * e - 3];
                const float y0 = __fsub_rn(__fmul_rn(x0, c[e]), __fmul_rn(x1, s[e]));
                const float y1 = __fadd_rn(__fmul_rn(x0, s[e]), __fmul_rn(x1, c[e]));
                if (e < 2) ya[2 * e] = y0, ya[2 * e + 1] = y1;
                else yb[2 * e - 4] = y0, yb[2 * e - 3] = y1;
            }
        }
        store4_from_f32(a.dst, db + d0, a.dst_dtype, ya);
        store4_from_f32(a.dst, db + d1, a.dst_dtype, yb);
    }
}
template <bool SMALL>
__device__ __forceinline__ void rope_rows_vec_types(const RopeRows &a, JobBlocks jb) {
    if (a.src_dtype == FHIP_F32) rope_rows_vec_body<SMALL, FHIP_F32>(a, jb);
    else if (a.src_dtype == FHIP_F16) rope_rows_vec_body<SMALL, FHIP_F16>(a, jb);
    else rope_rows_vec_body<SMALL, FHIP_BF16>(a, jb);
}
__device__ __forceinline__ void rope_rows_vec_any(const RopeRows &a, JobBlocks jb) {
    if (a.small) rope_rows_vec_types<true>(a, jb);
    else rope_rows_vec_types<false>(a, jb);
}

// The normalised variant on whole row blocks.  A lane holds four consecutive elements of a row; the sum of squares of a row
// is one lane's left-to-right fold (the order fixes the rounding), so the rows also pass through the wavefront's own LDS tile
// (pitch head_dim + 4 floats: the lanes then fold their rows without bank conflicts, four elements per read).  Every lane that
// has a row folds it, all lanes normalise what they hold, fetch the other halves of their pairs from the lanes that hold
// those, rotate and store.  The rows of a block are all read before any is written, so the destination may be the source.
// Bound: where blocks are few, one block's chain (fetch, fold, divide, store): so everything a block reads, the tables and
// weights included, is requested before it waits, and row numbers are divided by multiplication.  Where they are many,
// instructions and wavefronts per SIMD: squares are formed by all lanes and only added in the fold (half of its instructions), a row's
// elements are divided by way of its reciprocal, element types are known at compile time and bf16 is rounded by the hardware;
// blocks of 32 / 16 / 8 rows need more than the 128 registers of four wavefronts per SIMD.
// q, k and v of a layer, us a launch of a recorded graph, as before this and now: f32, 32/8 heads at 64, 512 rows 6.0 -> 5.7, 1000 9.1 -> 8.0; at
// 128, 512 rows 10.0 -> 8.1, 2000 25.6 -> 22.9; bf16 at 64, 100 rows 5.6 -> 4.6, 1000 10.4 -> 7.2; at 128, 100 rows 6.3 -> 5.1,
// 624 12.5 -> 8.8, 2000 27.8 -> 20.6.
constexpr int NORM_TILE_FLOATS = 1088;  // per wavefront: 16 rows of head_dim 64, 8 of 128, 4 of 256
constexpr int NORM_BLOCK_ROWS = 16;     // of a block at most
struct alignas(16) NormWaveLds {
    float tile[NORM_TILE_FLOATS];  // read and written in pieces of 16 bytes
    int64_t sb[NORM_BLOCK_ROWS], db[NORM_BLOCK_ROWS];  // element offsets of the block's rows in the source and the destination
    uint32_t pos[NORM_BLOCK_ROWS];                     // their positions (rows of the cos / sin tables, before pos0)
    float rms[NORM_BLOCK_ROWS], inv[NORM_BLOCK_ROWS];  // the rows' roots and their reciprocals
};
static_assert(offsetof(NormWaveLds, tile) % 16 == 0 && sizeof(NormWaveLds) % 16 == 0, "16-byte pieces of every wavefront's tile");
// value of x in the lane that holds the other half of this lane's pairs: CPR / 2 lanes away within the row's CPR lanes
template <int CPR>
__device__ __forceinline__ float other_half(float x) {
    const uint32_t u = __float_as_uint(x);
    if constexpr (CPR == 16) {
        return __uint_as_float(__builtin_amdgcn_update_dpp(0u, u, 0x128, 0xf, 0xf, true));  // row_ror:8
    } else if constexpr (CPR == 32) {
        const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        return __uint_as_float((threadIdx.x & 16) ? r[0] : r[1]);
    } else {
        const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        return __uint_as_float((threadIdx.x & 32) ? r[0] : r[1]);
    }
}
// x / d for the four elements of a lane, each correctly rounded.  inv = 1 / d to nearest: the quotient by it and one correction with
// the exact remainder is the quotient to nearest (Markstein, "Computation of elementary functions on the IBM RISC System/6000
// processor", 1990) where no step leaves the normal numbers; where an element or d might, the wavefront divides.
__device__ __forceinline__ float4_t divided_by(float4_t x, float d, float inv) {
    const float least = fminf(fminf(fabsf(x[0]), fabsf(x[1])), fminf(fabsf(x[2]), fabsf(x[3])));
    const float most = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3])));
    float4_t q;
    if (__builtin_amdgcn_ballot_w64(!(least >= 0x1p-80f && most <= 0x1p80f && d >= 0x1p-20f && d <= 0x1p20f)) == 0) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            q[e] = __fmul_rn(x[e], inv);
            q[e] = __builtin_fmaf(__builtin_fmaf(-q[e], d, x[e]), inv, q[e]);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) q[e] = __fdiv_rn(x[e], d);
    }
    return q;
}
// FEW: 32 / 16 / 8 rows at head_dim 64 / 128 / 256 divided by 2, or by 4 for inputs whose larger blocks would leave most SIMDs
// with one wavefront or none.
template <int D, int FEW, int SRC>
__device__ __forceinline__ void norm_rope_rows_vec_body(const RopeRows &a, NormWaveLds *w, JobBlocks jb) {
    constexpr int HALF = D / 2, CPR = D / 4, P = D + 4;
    static_assert(CPR <= 64 && 64 % CPR == 0 && D % 64 == 0, "head_dim 64, 128 or 256");
    // A wavefront step moves RS rows: lane -> (row SUB of the step, 16-byte piece C4 of the row).  A block is STEPS steps.
    constexpr int RS = 64 / CPR;
    constexpr int RPW = (D == 64 ? 32 : D == 128 ? 16 : 8) / FEW;  // rows per block
    constexpr int STEPS = RPW / RS;
    static_assert(RPW <= NORM_BLOCK_ROWS && RPW * P <= NORM_TILE_FLOATS && P % 4 == 0, "tile");
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float *tile = w->tile;
    const int sub = lane / CPR, c4 = lane % CPR;
    const int64_t rows = (int64_t)a.shape[0] * a.shape[1] * a.shape[2];
    const int64_t nblk = (rows + RPW - 1) / RPW;
    // cos and sin of this lane's elements: of pairs 4 c4 .. + 3 (halves: of the piece's place in its half), or of its two pairs
    const int ti = a.mode == 0 ? 4 * (c4 % (CPR / 2)) : 2 * c4;
    const bool heads_first = (a.few & NORM_HEADS_FIRST) != 0;
    for (int64_t blk = (int64_t)jb.at * 4 + wave; blk < nblk; blk += (int64_t)jb.count * 4) {
        const int64_t row0 = blk * RPW;
        const int nrow = (int)min((int64_t)RPW, rows - row0);
        if (lane < RPW) {
            const int64_t row = row0 + min(lane, nrow - 1);  // (lanes beyond the last row repeat it; nothing of theirs is stored)
            int64_t sb, db;
            uint32_t r;
            if (a.small) row_bases_small(a, (uint32_t)row, heads_first, &sb, &db, &r);
            else row_bases(a, row, heads_first, &sb, &db, &r);
            w->sb[lane] = sb, w->db[lane] = db, w->pos[lane] = r;
        }
        wave_lds_sync();
        Raw4<SRC> raw[STEPS];
        float4_t tc[STEPS], ts[STEPS];
#pragma unroll
        for (int u = 0; u < STEPS; u++) {
            const int lr = u * RS + sub;
            raw[u].load(a.src, w->sb[lr] + 4 * c4);
            tc[u] = float4_t{1.0f, 1.0f, 1.0f, 1.0f}, ts[u] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
            const int64_t at = (a.pos0 + w->pos[lr]) * HALF + ti;
            if (a.mode == 0) {
                tc[u] = *(const float4_t *)(a.cos + at), ts[u] = *(const float4_t *)(a.sin + at);
            } else if (a.mode == 1) {
                tc[u][0] = a.cos[at], tc[u][1] = a.cos[at + 1], ts[u][0] = a.sin[at], ts[u][1] = a.sin[at + 1];
            }
        }
        // weights (and bias) of this lane's elements: the same for every row
        float4_t wt, bias = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int e = 0; e < 4; e++) wt[e] = load_as_f32(a.norm_w, 4 * c4 + e, a.norm_dtype);
        if (a.norm_b) {
#pragma unroll
            for (int e = 0; e < 4; e++) bias[e] = load_as_f32(a.norm_b, 4 * c4 + e, a.norm_dtype);
        }
        // the squares, which are rounded before they are added
        float4_t x[STEPS];
#pragma unroll
        for (int u = 0; u < STEPS; u++) {
            x[u] = raw[u].widened();
            float4_t sq;
#pragma unroll
            for (int e = 0; e < 4; e++) sq[e] = __fmul_rn(x[u][e], x[u][e]);
            *(float4_t *)(tile + (u * RS + sub) * P + 4 * c4) = sq;
        }
        wave_lds_sync();
        if (lane < RPW) {
            float ss = 0.0f;
#pragma unroll 2
            for (int i = 0; i < D; i += 16) {  // sixteen values requested before the dependent chain consumes them
                float4_t v[4];
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = *(const float4_t *)(tile + lane * P + i + 4 * e);
#pragma unroll
                for (int e = 0; e < 16; e++) ss = __fadd_rn(ss, v[e >> 2][e & 3]);
            }
            // sqrtf is the correctly rounded root (the __fsqrt_rn intrinsic is the 1-ulp hardware approximation here)
            const float rms = sqrtf(__fadd_rn(__fdiv_rn(ss, (float)D), a.eps));
            w->rms[lane] = rms, w->inv[lane] = __fdiv_rn(1.0f, rms);
        }
        wave_lds_sync();
        // normalise, round to the tensor's type as the reference's norm does, rotate
#pragma unroll
        for (int u = 0; u < STEPS; u++) {
            const int lr = u * RS + sub;
            float4_t n = divided_by(x[u], w->rms[lr], w->inv[lr]), y;
#pragma unroll
            for (int e = 0; e < 4; e++) n[e] = __fmul_rn(n[e], wt[e]);
            if (a.norm_b) {
#pragma unroll
                for (int e = 0; e < 4; e++) n[e] = __fadd_rn(n[e], bias[e]);
            }
            n = rounded4<SRC>(n);
            if (a.mode == 2) {
                y = n;
            } else if (a.mode == 0) {
                const bool upper = c4 >= CPR / 2;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float o = other_half<CPR>(n[e]);
                    const float own = __fmul_rn(n[e], tc[u][e]), cross = __fmul_rn(o, ts[u][e]);
                    y[e] = __fadd_rn(own, upper ? cross : -cross);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const float x0 = n[2 * e], x1 = n[2 * e + 1];
                    y[2 * e] = __fsub_rn(__fmul_rn(x0, tc[u][e]), __fmul_rn(x1, ts[u][e]));
                    y[2 * e + 1] = __fadd_rn(__fmul_rn(x0, ts[u][e]), __fmul_rn(x1, tc[u][e]));
                }
            }
            if (lr < nrow) store4_from_f32(a.dst, w->db[lr] + 4 * c4, a.dst_dtype, y);
        }
        wave_lds_sync();  // the tile is rewritten by the next block
    }
}
template <int FEW, int SRC>
__device__ __forceinline__ void norm_rope_rows_vec_dims(const RopeRows &a, NormWaveLds *w, JobBlocks jb) {
    if (a.shape[3] == 128) norm_rope_rows_vec_body<128, FEW, SRC>(a, w, jb);
    else if (a.shape[3] == 256) norm_rope_rows_vec_body<256, FEW, SRC>(a, w, jb);
    else norm_rope_rows_vec_body<64, FEW, SRC>(a, w, jb);
}
template <int SRC>
__device__ __forceinline__ void norm_rope_rows_vec_few(const RopeRows &a, NormWaveLds *w, JobBlocks jb) {
    if ((a.few & NORM_FEW) == 4) norm_rope_rows_vec_dims<4, SRC>(a, w, jb);
    else norm_rope_rows_vec_dims<2, SRC>(a, w, jb);
}
__device__ __forceinline__ void norm_rope_rows_vec_any(const RopeRows &a, NormWaveLds *w, JobBlocks jb) {
    if (a.src_dtype == FHIP_F32) norm_rope_rows_vec_few<FHIP_F32>(a, w, jb);
    else if (a.src_dtype == FHIP_F16) norm_rope_rows_vec_few<FHIP_F16>(a, w, jb);
    else norm_rope_rows_vec_few<FHIP_BF16>(a, w, jb);
}

// The general form of the normalised variant (any strides): a workgroup takes groups of rows; one lane per row folds the squares in the
// reference's left-to-right order (the order fixes the rounding, so the sum is not split over lanes), the
// row's rms goes through LDS, then one lane per pair normalises and rotates as below.
constexpr int NORM_ROPE_MAX_ROWS = 256;
__device__ __forceinline__ void norm_rope_rows_body(const RopeRows &a, float *rms_of, JobBlocks jb) {
    const uint32_t D = a.shape[3], half = D / 2;
    const int64_t rows = (int64_t)a.shape[0] * a.shape[1] * a.shape[2];
    const int rpb = half >= 256 ? 1 : 256 / half;  // rows per group
    const int tid = threadIdx.x;
    for (int64_t row0 = (int64_t)jb.at * rpb; row0 < rows; row0 += (int64_t)jb.count * rpb) {
        const int nrow = (int)min((int64_t)rpb, rows - row0);
        if (tid < nrow) {
            int64_t t = row0 + tid;
            const uint32_t r = (uint32_t)(t % a.shape[2]);
            t /= a.shape[2];
            const int64_t sb = (t / a.shape[1]) * a.ss[0] + (t % a.shape[1]) * a.ss[1] + r * a.ss[2];
            float ss = 0.0f;
            for (uint32_t i = 0; i < D; i++) {
                const float x = load_as_f32(a.src, sb + i * a.ss[3], a.src_dtype);
                ss = __fadd_rn(ss, __fmul_rn(x, x));
            }
            // sqrtf is the correctly rounded root (the __fsqrt_rn intrinsic is the 1-ulp hardware approximation here)
            rms_of[tid] = sqrtf(__fadd_rn(__fdiv_rn(ss, (float)D), a.eps));
        }
        __syncthreads();  // also: every lane has read the row before any lane writes it (out may be x)
        for (int pidx = tid; pidx < nrow * (int)half; pidx += 256) {
            const int lr = pidx / half;
            const uint32_t i = pidx % half;
            int64_t t = row0 + lr;
            const uint32_t r = (uint32_t)(t % a.shape[2]);
            t /= a.shape[2];
            const int64_t sb = (t / a.shape[1]) * a.ss[0] + (t % a.shape[1]) * a.ss[1] + r * a.ss[2];
            const int64_t db = (t / a.shape[1]) * a.ds[0] + (t % a.shape[1]) * a.ds[1] + r * a.ds[2];
            const float rms = rms_of[lr];
            const uint32_t d0 = a.mode == 0 ? i : 2 * i, d1 = a.mode == 0 ? i + half : 2 * i + 1;
            float x0 = __fmul_rn(__fdiv_rn(load_as_f32(a.src, sb + d0 * a.ss[3], a.src_dtype), rms),
                                 load_as_f32(a.norm_w, d0, a.norm_dtype));
            float x1 = __fmul_rn(__fdiv_rn(load_as_f32(a.src, sb + d1 * a.ss[3], a.src_dtype), rms),
                                 load_as_f32(a.norm_w, d1, a.norm_dtype));
            if (a.norm_b) {
                x0 = __fadd_rn(x0, load_as_f32(a.norm_b, d0, a.norm_dtype));
                x1 = __fadd_rn(x1, load_as_f32(a.norm_b, d1, a.norm_dtype));
            }
            x0 = round_through(x0, a.src_dtype);
            x1 = round_through(x1, a.src_dtype);
            float y0 = x0, y1 = x1;
            if (a.mode != 2) {
                const float c = a.cos[(a.pos0 + r) * half + i], s = a.sin[(a.pos0 + r) * half + i];
                y0 = __fsub_rn(__fmul_rn(x0, c), __fmul_rn(x1, s));
                y1 = a.mode == 0 ? __fadd_rn(__fmul_rn(x1, c), __fmul_rn(x0, s))
                                 : __fadd_rn(__fmul_rn(x0, s), __fmul_rn(x1, c));
            }
            store_from_f32(a.dst, db + d0 * a.ds[3], a.dst_dtype, y0);
            store_from_f32(a.dst, db + d1 * a.ds[3], a.dst_dtype, y1);
        }
        __syncthreads();  // rms_of is rewritten by the next group
    }
}

// One normalised job.  6 vector registers and 12 bytes a lane lie in scratch; as one job of row_jobs_kernel, which spills none, the same
// launches take 1.03 of the time (us a launch of a recorded graph, before the present rows, so, and here, 32 heads: f32 at 64, 1000 rows 6.4, 6.8,
// 6.5; 128, 512 rows 7.2, 7.0, 6.7, 4096 34, 31, 29; bf16 at 128, 100 rows 6.1, 5.1, 4.8, 4096 37, 29, 28; 256, 1000 rows 21.5, 16.9, 16.3).
__global__ __launch_bounds__(256, 4) void norm_rope_rows_kernel(RopeRows a) {
    __shared__ NormWaveLds lds[4];
    __shared__ float rms_of[NORM_ROPE_MAX_ROWS];
    const JobBlocks jb = {blockIdx.x, gridDim.x};
    if (a.vec) norm_rope_rows_vec_any(a, &lds[threadIdx.x >> 6], jb);
    else norm_rope_rows_body(a, rms_of, jb);
}

__device__ __forceinline__ void rope_rows_body(const RopeRows &a, JobBlocks jb) {
    const uint32_t D = a.shape[3], half = D / 2;
    const int64_t per_row = a.mode == 2 ? D : half;
    const int64_t total = (int64_t)a.shape[0] * a.shape[1] * a.shape[2] * per_row;
    for (int64_t idx = (int64_t)jb.at * 256 + threadIdx.x; idx < total; idx += (int64_t)jb.count * 256) {
        const uint32_t i = (uint32_t)(idx % per_row);
        int64_t t = idx / per_row;
        const uint32_t r = (uint32_t)(t % a.shape[2]);
        t /= a.shape[2];
        const uint32_t h = (uint32_t)(t % a.shape[1]);
        const uint32_t b = (uint32_t)(t / a.shape[1]);
        const int64_t sb = b * a.ss[0] + h * a.ss[1] + r * a.ss[2];
        const int64_t db = b * a.ds[0] + h * a.ds[1] + r * a.ds[2];
        if (a.mode == 2) {
            store_from_f32(a.dst, db + i * a.ds[3], a.dst_dtype, load_as_f32(a.src, sb + i * a.ss[3], a.src_dtype));
            continue;
        }
        const float c = a.cos[(a.pos0 + r) * half + i], s = a.sin[(a.pos0 + r) * half + i];
        const uint32_t d0 = a.mode == 0 ? i : 2 * i, d1 = a.mode == 0 ? i + half : 2 * i + 1;
        const float x0 = load_as_f32(a.src, sb + d0 * a.ss[3], a.src_dtype);
        const float x1 = load_as_f32(a.src, sb + d1 * a.ss[3], a.src_dtype);
        // every product and sum is rounded on its own: this file is compiled with -ffp-contract=off
        const float y0 = __fsub_rn(__fmul_rn(x0, c), __fmul_rn(x1, s));
        const float y1 = a.mode == 0 ? __fadd_rn(__fmul_rn(x1, c), __fmul_rn(x0, s))
                                     : __fadd_rn(__fmul_rn(x0, s), __fmul_rn(x1, c));
        store_from_f32(a.dst, db + d0 * a.ds[3], a.dst_dtype, y0);
        store_from_f32(a.dst, db + d1 * a.ds[3], a.dst_dtype, y1);
    }
}

// Eight wavefronts per SIMD: bound by how many loads are on their way (f32, 16384 rows of 32 heads at 128: 207 us with seven,
// which 101 scalar registers allow, 196 with eight).
__global__ __launch_bounds__(256, 8) void rope_rows_kernel(RopeRows a) {
    const JobBlocks jb = {blockIdx.x, gridDim.x};
    if (a.vec) rope_rows_vec_any(a, jb);
    else rope_rows_body(a, jb);
}

// Several row jobs in one launch, each with workgroups of its own: the rotation of q, the rotated keys and the values of
// one decode step are three tiny jobs whose launch cost exceeds their run time.
__global__ __launch_bounds__(256, 4) void row_jobs_kernel(RowJobs js) {
    __shared__ NormWaveLds lds[4];
    __shared__ float rms_of[NORM_ROPE_MAX_ROWS];
    const uint32_t wg = blockIdx.x;
    const int j = wg >= js.first[1] ? (wg >= js.first[2] ? 2 : 1) : 0;
    const uint32_t from = j == 0 ? 0u : js.first[j], end = j == 0 ? js.first[1] : j == 1 ? js.first[2] : gridDim.x;
    // (by way of the arguments' own address: the compiler would copy a struct that it indexes to the stack)
    static_assert(offsetof(RowJobs, job) == 0, "the jobs come first");
    const RopeRows &a = *(const RopeRows *)((const __attribute__((address_space(4))) RopeRows *)__builtin_amdgcn_kernarg_segment_ptr() + j);
    const JobBlocks jb = {wg - from, end - from};
    if (a.norm_w) {
        if (a.vec) norm_rope_rows_vec_any(a, &lds[threadIdx.x >> 6], jb);
        else norm_rope_rows_body(a, rms_of, jb);
    } else {
        if (a.vec) rope_rows_vec_any(a, jb);
        else rope_rows_body(a, jb);
    }
}

// Blocks of the wide normalised form for the jobs of one launch (see norm_rope_rows_vec_body).  A quarter of 32 / 16 / 8 rows while
// nearly all of the wavefronts are resident at once (four per SIMD of a 256-CU chip; us a launch, quarters and halves: f32, 32/8
// heads at 64, 624 rows 6.2 and 6.4, 1000 9.3 and 7.8; at 128, 250 rows 6.0 and 6.7, 512 9.6 and 8.5), half of them beyond.  Halves take the heads of
// a position together where those are neighbours in the source (f32, 32/8 heads at 128, 2000 rows 24.7 -> 22.9).
static void choose_norm_blocks(RopeRows *jobs, int n) {
    int64_t blocks = 0;
    for (int i = 0; i < n; i++) {
        const RopeRows &a = jobs[i];
        if (!a.norm_w || !a.vec) continue;
        const int64_t rows = (int64_t)a.shape[0] * a.shape[1] * a.shape[2], quarter = a.shape[3] == 64 ? 8 : a.shape[3] == 128 ? 4 : 2;
        blocks += (rows + quarter - 1) / quarter;
    }
    for (int i = 0; i < n; i++)
        jobs[i].few = blocks < 3584 ? 4 : jobs[i].ss[1] < jobs[i].ss[2] ? 2 | NORM_HEADS_FIRST : 2;
}

void fill_row_job(RopeRows *out, const void *src, const int64_t ss[4], fhip_dtype src_dtype, void *dst, const int64_t ds[4],
                  fhip_dtype dst_dtype, const uint32_t shape[4], const float *cos, const float *sin, int64_t pos0, int mode,
                  const RowNorm *norm) {
    RopeRows &a = *out;
    a.src = src;
    a.dst = dst;
    for (int i = 0; i < 4; i++) {
        a.ss[i] = ss[i];
        a.ds[i] = ds[i];
        a.shape[i] = shape[i];
    }
    a.src_dtype = src_dtype;
    a.dst_dtype = dst_dtype;
    a.cos = cos;
    a.sin = sin;
    a.pos0 = pos0;
    a.mode = mode;
    a.norm_w = norm ? norm->weight : nullptr;
    a.norm_b = norm ? norm->bias : nullptr;
    a.norm_dtype = norm ? norm->dtype : FHIP_F32;
    a.eps = norm ? norm->eps : 0.0f;
    // the wide forms: consecutive elements, every row start a multiple of four elements from an address aligned to
    // four elements, on both sides; the tables (if used) 16-byte aligned
    const uint32_t D = shape[3];
    auto wide = [&](const void *p, const int64_t st[4], fhip_dtype t) {
        const uintptr_t step = (t == FHIP_F32 ? 4 : 2) * 4;
        if (D > 1 && st[3] != 1) return false;
        if (((uintptr_t)p % step) != 0) return false;
        for (int i = 0; i < 3; i++)
            if (shape[i] > 1 && st[i] % 4 != 0) return false;
        return true;
    };
    a.vec = D % 8 == 0 && D >= 8 && wide(src, ss, src_dtype) && wide(dst, ds, dst_dtype) &&
            (mode == 2 || (((uintptr_t)cos % 16) == 0 && ((uintptr_t)sin % 16) == 0));
    if (a.norm_w && !(D == 64 || D == 128 || D == 256)) a.vec = 0;  // the head dims the wide normalised form is built for
    // Division by multiplication: with 2^(l - 1) < d <= 2^l and mul = floor(2^(31 + l) / d) + 1 (below 2^32), mul d is 2^(31 + l)
    // and at most d <= 2^l more, so t mul / 2^(31 + l) is t / d and less than 1 / d more for t < 2^31.
    const uint32_t divisors[3] = {shape[2], shape[1], mode == 2 ? D / 4 : D / 8};
    for (int i = 0; i < 3; i++) {
        const uint32_t d = divisors[i];
        int l = 0;
        while (l < 32 && ((uint64_t)1 << l) < d) l++;
        a.mul[i] = d > 1 && l < 32 ? (uint32_t)(((uint64_t)1 << (31 + l)) / d + 1) : 0;
        a.shift[i] = l > 0 ? l - 1 : 0;
    }
    const unsigned __int128 steps = (unsigned __int128)shape[0] * shape[1] * shape[2] * (norm ? 1 : divisors[2] ? divisors[2] : 1);
    a.small = steps < (1u << 31);
    a.few = 4;
    choose_norm_blocks(out, 1);
}

// rows per wavefront block of the wide normalised form (RPW in norm_rope_rows_vec_body)
static int norm_rows_per_wave(const RopeRows &a) {
    const int D = (int)a.shape[3];
    return (D == 64 ? 32 : D == 128 ? 16 : 8) / (a.few & NORM_FEW);
}

static int64_t job_blocks(const RopeRows &a) {
    const int64_t rows = (int64_t)a.shape[0] * a.shape[1] * a.shape[2];
    if (rows == 0 || a.shape[3] == 0) return 0;
    if (a.norm_w) {
        const int rpb = a.vec ? 4 * norm_rows_per_wave(a) : (a.shape[3] / 2 >= 256 ? 1 : 256 / (a.shape[3] / 2));
        return (rows + rpb - 1) / rpb;
    }
    const int64_t total = a.vec ? rows * (a.mode == 2 ? a.shape[3] / 4 : a.shape[3] / 8)
                                : rows * (a.mode == 2 ? a.shape[3] : a.shape[3] / 2);
    return (total + 255) / 256;
}

int launch_row_jobs(const RowJobs &given, hipStream_t stream) {
    RowJobs js = given;
    choose_norm_blocks(js.job, js.n);
    uint32_t blocks = 0;
    for (int i = 0; i < 3; i++) {
        js.first[i] = blocks;
        const int64_t need = i < js.n ? job_blocks(js.job[i]) : 0;
        blocks += (uint32_t)(need < 65536 ? need : 65536);  // (a job's workgroups stride over its work)
    }
    if (blocks == 0) return FHIP_OK;
    hipLaunchKernelGGL(row_jobs_kernel, dim3(blocks), dim3(256), 0, stream, js);
    FHIP_HIP_CHECK(hipGetLastError());
    return FHIP_OK;
}

int launch_rope_rows(const void *src, const int64_t ss[4], fhip_dtype src_dtype, void *dst, const int64_t ds[4],
                     fhip_dtype dst_dtype, const uint32_t shape[4], const float *cos, const float *sin, int64_t pos0,
                     int mode, const RowNorm *norm, hipStream_t stream) {
    RopeRows a;
    fill_row_job(&a, src, ss, src_dtype, dst, ds, dst_dtype, shape, cos, sin, pos0, mode, norm);
    const int64_t blocks = job_blocks(a);
    if (blocks == 0) return FHIP_OK;
    const dim3 grid((unsigned)(blocks < 65536 ? blocks : 65536));
    if (a.norm_w) hipLaunchKernelGGL(norm_rope_rows_kernel, grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL(rope_rows_kernel, grid, dim3(256), 0, stream, a);
    FHIP_HIP_CHECK(hipGetLastError());
    return FHIP_OK;
}

}  // namespace fhip
