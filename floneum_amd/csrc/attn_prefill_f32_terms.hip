// Prefill attention in f32 precision on the 16-bit matrix cores (v_mfma_f32_32x32x16_bf16).
//
// The f32 matrix instruction runs at a sixteenth of the bf16 one's rate.  An f32 value is the exact sum of three bf16
// terms (8 significant bits each: x = t0 + t1 + t2, each term what rounding the rest to bf16 leaves), so a product of two
// f32 values is the sum of nine products of terms, each exact in the f32 accumulator's input.  The three smallest (t1 t2,
// t2 t1, t2 t2) are below 2^-24 of the product in the worst case and 2^-27 of it in the mean, less than one rounding of
// the f32 accumulation; the other six are formed: 6 / 16 of the f32 instruction's matrix time.  16-bit tensors, which
// this kernel serves where their own one does not (finite mask values), have two terms (f16) or one (bf16); the
// probabilities are f32 values and always have three.
// Infinities: an element of Q, K or V that is +-inf (or beyond 3.39e38, bf16's largest) makes its products NaN.
// Small elements: below 2^-110 the last bits of a value fall below bf16's smallest number, 2^-133, and its terms are off by up to
// 2^-134.  That is nothing beside a result of 2^-110 and more, and nothing in a score unless the other factor is beyond 2^100.
// Rows whose sums are not finite or smaller than that at the end, and rows with elements of (scaled) Q beyond either limit,
// are formed once more without terms (unit_in_f32).  What is left: a probability below 2^-110 counts to 2^-134 only, which
// shows where V's elements are 2^110 times the result, and results of elements below 2^-134 are zero.
//
// A unit is 32 query rows of one head; a wavefront owns one.  A workgroup holds U units that share a KV head (the heads of
// a GQA group first, then further rows) and walks the keys they see in tiles of 32 rows, which are split into terms on the
// way into LDS (11 vector instructions per two elements, once per workgroup) and kept there as bf16 planes.
//   S^T (32 keys x 32 queries) = K_tile . Q^T    A = K[key][dim] from LDS, B = Q's terms, in registers for the whole kernel
//   softmax down the key axis as in attn_prefill_mfma.hip: probabilities against the row's reference exponent, which
//   moves only when a lane's probabilities of a tile sum to more than 2^15
//   O^T (D x 32 queries) += V^T . P^T            A = V^T by transposing LDS reads of the row-major planes,
//                                                B = the terms of the S^T accumulator registers themselves
// Scores sum the products of leading terms and all others in two accumulators, and a tile's share of O^T forms on its own
// and is added once: few roundings happen at the size of the result (relative error of a 4096-token prompt against 64 bits
// 6.9e-8; f32 matrix instructions 2.2e-7).
// K and V take turns in one set of staging registers (V(t) is in flight under S^T(t), K(t + 1) under P.V(t)) but have
// their own LDS image; two barriers per tile.  With KG > 1 the workgroup has KG times the wavefronts: group g takes the
// tiles t with t % KG == g through its own LDS image, and the groups' states are merged at the end.
//
// Bound: f32 4096 x 4096 causal, 32/8 heads, D = 128, 670 - 700 us (1150 on the f32 matrix instruction) = 205 TFLOP/s of
// f32 products or 1.23 PFLOP/s of bf16 ones, 73 % of what the matrix cores alone sustain on random bf16 operands under the
// power limit.  The matrix pipes are busy 67 % of the cycles at 1.7 GHz; all-zero inputs (no toggling, 2.4 GHz) take 563
// us.  A tile is 96 matrix instructions (D = 128, 3072 cycles) and about 390 vector ones per wavefront (splitting K and V
// 176, the probabilities 88, softmax 50, the additions of O 64).
//
// Reference semantics: fusor-ml/fusor/src/composite/flash_attention.rs:141-199; f32 is the data type kalosm-llama always
// calls with (models/kalosm-llama/src/raw/attention_layer.rs:400-448).
#include <algorithm>

#include "attn_bounds.h"
#include "attn_f32.h"
#include "common.h"
#include "device_utils.h"

namespace fhip {

constexpr int PT_BN = 32;  // keys per tile
typedef float4_t __attribute__((aligned(8))) float4_at8_t;  // a row of the partials is D + 2 floats
constexpr int SCAN_KEYS = 1024;  // longest mask row a wavefront looks at itself

#define LDST_PTR(type, byte_off) ((__attribute__((address_space(3))) type *)(lds_base + (byte_off)))

template <typename T>
struct Terms {
    static constexpr int N = 3;
};
template <>
struct Terms<half_t> {
    static constexpr int N = 2;
};
template <>
struct Terms<bf16_t> {
    static constexpr int N = 1;
};

// Four values as N bf16 terms each: term i of (x0, x1) packed into lo[i], of (x2, x3) into hi[i], each term what rounding
// the rest to bf16 (to nearest even) leaves.  In assembly, because the compiler converts what it has converted once more for
// the rest, and leaves each pair's chain of dependent instructions in a row.
template <int N>
__device__ __forceinline__ void split4(float4_t x, uint32_t (&lo)[N], uint32_t (&hi)[N]) {
#pragma unroll
    for (int i = 0; i < N; i++) {
        if (i + 1 == N) {
            asm("v_cvt_pk_bf16_f32 %0, %2, %3\n\t"
                "v_cvt_pk_bf16_f32 %1, %4, %5"
                : "=&v"(lo[i]), "=v"(hi[i])
                : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]));
        } else {
            float4_t rest;
            asm("v_cvt_pk_bf16_f32 %0, %6, %7\n\t"
                "v_cvt_pk_bf16_f32 %1, %8, %9\n\t"
                "v_lshlrev_b32 %2, 16, %0\n\t"
                "v_and_b32 %3, 0xffff0000, %0\n\t"
                "v_lshlrev_b32 %4, 16, %1\n\t"
                "v_and_b32 %5, 0xffff0000, %1\n\t"
                "v_sub_f32 %2, %6, %2\n\t"
                "v_sub_f32 %3, %7, %3\n\t"
                "v_sub_f32 %4, %8, %4\n\t"
                "v_sub_f32 %5, %9, %5"
                : "=&v"(lo[i]), "=&v"(hi[i]), "=&v"(rest[0]), "=&v"(rest[1]), "=&v"(rest[2]), "=&v"(rest[3])
                : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]));
            x = rest;
        }
    }
}

constexpr float SMALLEST_IN_TERMS = 0x1p-110f, LARGEST_Q = 0x1p100f;
// orders values by their magnitude, with zero above all
__device__ __forceinline__ uint32_t magnitude(float x) { return (__float_as_uint(x) << 1) - 1; }

// four elements at a byte offset of a buffer, as f32
template <typename T>
__device__ __forceinline__ float4_t buffer_load4(__amdgpu_buffer_rsrc_t rows, int at, int from) {
    if constexpr (sizeof(T) == 4) {
        return __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(rows, at, from, 0));
    } else {
        const auto raw = __builtin_amdgcn_raw_buffer_load_b64(rows, at, from, 0);
        return load4((const T *)&raw);
    }
}

template <typename T>
__device__ __forceinline__ float buffer_load1(__amdgpu_buffer_rsrc_t rows, int at, int from) {
    if constexpr (sizeof(T) == 4) return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rows, at, from, 0));
    else return to_float(__builtin_bit_cast(T, (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rows, at, from, 0)));
}

// U: units per workgroup, KG: key groups (wavefronts = U * KG)
template <typename T, int D, int U>
struct PtCfg {
    static constexpr int N = Terms<T>::N;
    // K rows 16 bytes apart modulo the 256-byte bank period (16-byte reads of 16 rows); V rows 64 bytes apart (the
    // transposing read of 4 rows x 64 bytes)
    static constexpr int KP = D * 2 + 16;
    static constexpr int VP = D * 2 + (D * 2 % 128 == 0 ? 64 : 0);
    static constexpr int K_PLANE = PT_BN * KP, V_PLANE = PT_BN * VP;
    static constexpr int V_BASE = N * K_PLANE;
    static constexpr int G_BYTES = N * (K_PLANE + V_PLANE);  // one key group's tile
    static constexpr int GT = 64 * U;  // threads of a key group, which move its tiles
    // A wavefront's rows of Q and of the result pass through LDS, so that memory sees whole lines: half of Q's dims and 32
    // dims of the result at a time, in the space of the tiles.
    static constexpr int HALF_PITCH = D * 2 + 16, OUT_PITCH = 32 * 4 + 16;
    static constexpr int ROWS_BYTES = 32 * (HALF_PITCH > OUT_PITCH ? HALF_PITCH : OUT_PITCH);
    static constexpr int CPR = D / 4;  // pieces of four elements per row
    // lanes per row and, between a thread's pieces, rows or columns: whole rows where they divide the threads
    static constexpr int LPR = GT % CPR == 0 ? CPR : 8;
    static constexpr int RSTEP = GT / LPR;  // rows a group moves at once
    static constexpr int CSTEPS = CPR / LPR;
    static constexpr int NCH = PT_BN * CPR / GT;
};

// What the launcher works out for the kernel.
struct TermsLaunch {
    uint32_t g_magic;  // unit / G = (unit * g_magic) >> 32 (0: G is 1)
    int32_t snake;     // workgroups from this one of the last grid dimension on are numbered backwards (0: none)
    int32_t out_vec;   // bytes per store of the result: 16 (f32), 8 (16-bit), or 0: element by element
    int32_t mask_rows; // an added mask is read four keys at a time through a buffer
    int32_t level_pitch;  // uneven shares: workgroups per KV head that a share's keys are ahead of the next one's (0: the grid's order)
};

// K, V and Q of a unit as buffers: bytes from row to row, and where this lane's row of Q begins
struct RowBuffers {
    __amdgpu_buffer_rsrc_t k, v, q;
    int k_bytes, v_bytes, q_at;
};

// A wavefront's unit in f32 arithmetic (v_mfma_f32_32x32x2_f32), for units with rows that met an element without finite bf16
// terms: references, sums (this half's keys) and unnormalised results as the kernel holds them.  K and V come straight from
// memory, a wavefront's tile at a time.  Keys that a row does not see must not reach it (0 x inf is NaN): where some row sees a
// tile in part and V's 32 dims of it are not finite, they are taken key by key.  mine: 4 KiB of LDS of this wavefront's; mrow:
// this lane's mask values to add, or NULL; rows: those that matter, and once they are all NaN nothing more is formed.
// Bound: the f32 matrix instruction, and memory latency where few wavefronts are left.  An infinity in V at the first key, so
// that every unit comes here (us, without it in brackets; one row at a time before): 4096 causal rows of 32/8 heads, D = 128
// 2250 (740; 86800), 512 rows at D = 64 81 (21.5; 4230), 129 rows on 8003 keys 418 (131; 22000).
template <typename T, int D>
__device__ __forceinline__ void unit_in_f32(const AttnParams &p, __attribute__((address_space(3))) char *mine, const RowBuffers &rows_of,
                                            const T *mrow, const RowBounds &rb, uint32_t rows, int lane, float16_t (&o)[D / 32], float &m,
                                            float &l) {
    constexpr int NDB = D / 32, ES = sizeof(T);
    const int ln = lane & 31, h2 = lane >> 5;
    auto uniform = [](int x) __attribute__((always_inline)) { return __builtin_amdgcn_readfirstlane(x); };
    const int lo_w = uniform(rb.lo_w), hi_w = uniform(rb.hi_w), full_lo_w = uniform(rb.full_lo_w), full_hi_w = uniform(rb.full_hi_w);
    const float log2_unit = mrow ? PF32_LOG2E : 1.0f, score_scale = mrow ? p.scale : p.scale * PF32_LOG2E;
    auto p_lds = (__attribute__((address_space(3))) float *)mine;  // [key][query] of a tile seen in part
    m = -INFINITY, l = 0.0f;
#pragma unroll
    for (int db = 0; db < NDB; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[db][r] = 0.0f;
#pragma unroll 1
    for (int tile = lo_w / PT_BN; tile * PT_BN < hi_w; tile++) {
        int j0 = tile * PT_BN;
        asm volatile("" : "+s"(j0));  // (no address of the body is carried from tile to tile: they would not fit the registers)
        float16_t s;
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = 0.0f;
#pragma unroll 1
        for (int d0 = 0; d0 < D; d0 += 32) {
            float4_t kr[4], qr[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int dim = d0 + 8 * i + 4 * h2, none = dim < p.D ? 0 : (int)0x80000000;
                kr[i] = buffer_load4<T>(rows_of.k, (ln * rows_of.k_bytes + dim * ES) | none, j0 * rows_of.k_bytes);
                qr[i] = buffer_load4<T>(rows_of.q, (rows_of.q_at + dim * ES) | none, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[i][e], qr[i][e], s, 0, 0, 0);
        }
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int key = j0 + 8 * (r >> 2) + 4 * h2 + (r & 3);
            const bool seen = key >= rb.klo && key < rb.khi;
            const float x = mrow ? __builtin_fmaf(s[r], score_scale, seen ? to_float(mrow[key * p.ms1]) : 0.0f) : s[r] * score_scale;
            s[r] = seen ? x : -INFINITY;
            mx = fmaxf(mx, s[r]);  // (passes NaN by: such a score leaves the reference alone and makes the sums NaN)
        }
        const float m_new = fmaxf(m, half_swap_max32(mx)), corr = moved_reference(m, m_new, log2_unit);
        m = m_new;
        l *= corr;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            s[r] = probability(s[r], m, log2_unit);
            l += s[r];
        }
#pragma unroll
        for (int db = 0; db < NDB; db++) o[db] *= corr;
        // (dims behind head_dim hold whatever follows, and are not written)
        const bool full = j0 >= full_lo_w && j0 + PT_BN <= full_hi_w;
        if (!full) {
            wave_lds_sync();
#pragma unroll
            for (int r = 0; r < 16; r++) p_lds[(8 * (r >> 2) + 4 * h2 + (r & 3)) * 32 + ln] = s[r];
            wave_lds_sync();
        }
#pragma unroll
        for (int db = 0; db < NDB; db++) {
            float a[16], zero = 0.0f;
            const int at = 4 * h2 * rows_of.v_bytes + (32 * db + ln) * ES;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                a[r] = buffer_load1<T>(rows_of.v, at, (j0 + 8 * (r >> 2) + (r & 3)) * rows_of.v_bytes);
                zero = __builtin_fmaf(a[r], 0.0f, zero);
            }
            if (full || __builtin_amdgcn_ballot_w64(!(zero == 0.0f)) == 0) {
                // this tile's share on its own, then one addition at the size of the sum
                float16_t sum;
#pragma unroll
                for (int r = 0; r < 16; r++) sum[r] = 0.0f;
#pragma unroll
                for (int r = 0; r < 16; r++) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(a[r], s[r], sum, 0, 0, 0);
                o[db] += sum;
            } else {
                const int end = min(j0 + PT_BN, hi_w);
#pragma unroll 1
                for (int key = max(j0, lo_w); key < end; key++) {
                    const float w = p_lds[(key - j0) * 32 + ln];
                    const bool seen = key >= rb.klo && key < rb.khi;
#pragma unroll
                    for (int rq = 0; rq < 4; rq++) {
                        const float4_t x = buffer_load4<T>(rows_of.v, (32 * db + 8 * rq + 4 * h2) * ES, key * rows_of.v_bytes);
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            o[db][4 * rq + e] = seen ? __builtin_fmaf(w, x[e], o[db][4 * rq + e]) : o[db][4 * rq + e];
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);  // (16 loads at a time)
        }
        const uint64_t nan = __builtin_amdgcn_ballot_w64(l != l);
        if ((((uint32_t)nan | (uint32_t)(nan >> 32)) & rows) == rows) return;
    }
}

template <typename T, int D, int U, int KG, int MODE>
__global__ __launch_bounds__(64 * U * KG, D > 128 || (KG == 2 && U == 2 && D > 64) ? 1 : KG == 1 && D == 64 && MODE == PF32_INTERVALS ? 3 : 2) void prefill_f32_terms_kernel(AttnParams p, TermsLaunch tl) {
    typedef PtCfg<T, D, U> C;
    constexpr int N = C::N, NDB = D / 32, NKB = D / 16;
    constexpr bool BIAS = MODE != PF32_INTERVALS;
    // Which phase of the two wavefronts on a SIMD goes first where both could issue: the matrix one at wide heads, the vector
    // one where a tile's matrix work is short beside it.  D = 64: 12 x 700 rows with added masks 127 us without priorities,
    // 126 / 122 with the matrix / vector phase first, 2048-row prompt 115, 112 / 110.5; D = 128: 1024-row prompt 79, 76 / 76,
    // 4096 rows 717, 711 / 718.
    // Four key groups (few tiles per wavefront) gain nothing from the vector phase: 512-row layer 29.3 against 29.7.
    constexpr int MATRIX_PRIO = D > 64 || KG == 4 ? 1 : 0;
    __shared__ __attribute__((aligned(16))) char smem[KG * C::G_BYTES > U * KG * C::ROWS_BYTES ? KG * C::G_BYTES : U * KG * C::ROWS_BYTES];
    auto lds_base = (__attribute__((address_space(3))) char *)smem;

    // The arguments are requested together: read where they are used, between branches, they cost a short call a memory
    // latency each.
    pin(p.q, p.k, p.v, p.out, p.mask, p.kv_lens, p.qs[0], p.qs[1], p.qs[2], p.ks[0], p.ks[1], p.ks[2]);
    pin(p.vs[0], p.vs[1], p.vs[2], p.os[0], p.os[1], p.os[2], p.ms0, p.B, p.Hkv, p.G, p.Sq, p.Skv, p.D, p.mask_kind);
    pin(p.analytic, p.causal, p.q_pos_offset, p.window, p.scale, p.iv, p.iv_bad, p.only_if_bad, p.bad_tag, p.pf_nsplit, p.pf_chunk,
        p.iv_either, tl.g_magic, tl.snake, tl.mask_rows);

    if constexpr (MODE == PF32_BIAS) {
        if (p.only_if_bad && *p.only_if_bad != p.bad_tag) return;  // the interval form of the mask has served the call
    } else if constexpr (MODE == PF32_INTERVALS) {
        if (p.iv_bad && *p.iv_bad == p.bad_tag) return;  // the mask is not made of intervals: the BIAS form takes the call
    }
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int ln = lane & 31;
    const int h2 = lane >> 5;

    const int grp = wave / U;       // key group
    const int gtid = tid % C::GT;   // thread inside the group
    const int gbase = grp * C::G_BYTES;

    // Workgroup -> (units, batch, kv head): the units of a KV head are its row blocks times the query heads that share it,
    // numbered heads first, so that U consecutive ones read the same keys; those with the most keys first.
    // (grid: shares of the keys, kv heads of the batch, workgroups per kv head)
    const int nks = gridDim.x, nwg = gridDim.z;
    int ksplit = blockIdx.x, rem = blockIdx.y, wz = blockIdx.z;
    // The shares of a square prompt differ in length: workgroup wz + P of a share sees as many keys of it as workgroup wz of the next
    // one (P: level_pitch), so those with equal wz + share * P are a level, and the levels are numbered the longest first, without gaps.
    // Workgroups are dealt to the shader engines in turn, which a descending order evens out.  us at head_dim 256, in the grid's order
    // turned with wz and its plan, and now: 1300 rows of 12/12 heads 141 -> 111, 2000 of 16/4 347 -> 235, 800 of 32/8 151 -> 105.
    if constexpr (D > 128) {
        if (tl.level_pitch) {
            const int id = (wz * gridDim.y + rem) * nks + ksplit, pitch = tl.level_pitch;
            int t = id / (int)gridDim.y, level = 0, first = 0, end = 1;  // shares first .. end - 1 have workgroups in this level
            rem = id - t * (int)gridDim.y;
            for (;;) {
                const int start = end < nks ? end * pitch : 0x7fffffff, stop = first * pitch + nwg, next = min(start, stop);
                const int shares = end - first, here = (next - level) * shares;
                if (t < here) {
                    level += t / shares;
                    ksplit = first + t % shares;
                    break;
                }
                t -= here;
                level = next;
                end += next == start;
                first += next == stop;
            }
            wz = level - ksplit * pitch;
        }
    }
    // with the whole grid resident at once (two workgroups per CU) a CU gets a long and a short one
    const int wg = tl.snake > 0 && wz >= tl.snake ? tl.snake + nwg - 1 - wz : wz;
    const int first_unit = (nwg - 1 - wg) * U;
    auto over_g = [&](int u) __attribute__((always_inline)) { return tl.g_magic ? (int)__umulhi((uint32_t)u, tl.g_magic) : u; };
    const int b = p.B > 1 ? rem / p.Hkv : 0;
    int g = rem - b * p.Hkv;
    if ((p.Hkv & 7) == 0) g = (g & 7) * (p.Hkv >> 3) + (g >> 3);  // workgroups of one XCD share KV heads
    const int unit = first_unit + wave % U;
    const int unit_row = over_g(unit);  // 32-row block of the unit
    const int h = g * p.G + unit - unit_row * p.G;
    // rows of a tile beyond the sequence's own keys, or behind the last query's position, are never fetched (what they
    // hold, NaN included, must not reach the result as 0 x NaN in P . V)
    int key_end = p.kv_lens ? min(p.Skv, max(p.kv_lens[b], 1)) : p.Skv;
    if (p.analytic && p.causal) key_end = (int)min((int64_t)key_end, max(p.q_pos_offset + p.Sq, (int64_t)1));

    const int q0 = 32 * over_g(first_unit);                      // first row of the workgroup
    const int bm = 32 * (over_g(first_unit + U - 1) + 1) - q0;   // rows from there to its last
    const int qw0 = 32 * unit_row;
    const int query = qw0 + ln;
    // uniform over the sequence
    bool bias_on = MODE == PF32_BIAS;
    int2 span = {0, 0x7fffffff};
    if constexpr (MODE == PF32_EITHER) {
        if (p.iv_either == 2) {
            // What the scan launch would find, of this sequence's row alone (at most SCAN_KEYS keys, in whole pieces): that
            // launch in front cost 8 x 512 keys 4.7 us, the row's pieces come in about the time its result took to read.
            const auto row = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.mask + b * p.ms0), 0, p.Skv * (int)sizeof(T), 0x00020000);
            constexpr int PIECES = SCAN_KEYS / 256;
            float4_t x[PIECES];
#pragma unroll
            for (int i = 0; i < PIECES; i++)
                if (256 * i < p.Skv) x[i] = buffer_load4<T>(row, lane * 4 * (int)sizeof(T), 256 * i * (int)sizeof(T));
            int lo = 0x7fffffff, hi = 0, zeros = 0;
            bool others = false;
#pragma unroll
            for (int i = 0; i < PIECES; i++) {
                if (256 * i >= p.Skv) continue;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int key = 256 * i + 4 * lane + e;
                    const bool zero = key < p.Skv && x[i][e] == 0.0f;
                    others |= key < p.Skv && !zero && x[i][e] != -INFINITY;
                    lo = zero ? min(lo, key) : lo;
                    hi = zero ? key + 1 : hi;
                    zeros += zero;
                }
            }
            lo = wave_reduce_i(lo, [](int x, int y) { return min(x, y); });
            hi = wave_reduce_i(hi, [](int x, int y) { return max(x, y); });
            zeros = wave_reduce_i(zeros, [](int x, int y) { return x + y; });
            if (zeros == 0) lo = 0;  // no visible key: the empty interval
            bias_on = __builtin_amdgcn_ballot_w64(others) != 0 || __builtin_amdgcn_readfirstlane(zeros) != __builtin_amdgcn_readfirstlane(hi - lo);
            if (!bias_on) span = {lo, hi};
        } else {
            bias_on = *p.iv_bad == p.bad_tag;
        }
    }
    RowBounds rb = row_bounds(p, MODE == PF32_BIAS ? nullptr : p.iv, b, q0, bm, qw0, lane, span);
    if constexpr (MODE == PF32_EITHER) {
        if (bias_on) rb = row_bounds(p, nullptr, b, q0, bm, qw0, lane);
    }
    if (nks > 1) {  // this workgroup's share of the keys
        const int c_lo = ksplit * p.pf_chunk, c_hi = c_lo + p.pf_chunk;
        rb.lo_wg = max(rb.lo_wg, c_lo), rb.hi_wg = min(rb.hi_wg, c_hi);
        rb.lo_w = max(rb.lo_w, c_lo), rb.hi_w = min(rb.hi_w, c_hi);
        rb.full_lo_w = max(rb.full_lo_w, c_lo), rb.full_hi_w = min(rb.full_hi_w, c_hi);
        rb.klo = max(rb.klo, c_lo), rb.khi = min(rb.khi, c_hi);
    }
    // uniform values, kept in scalar registers
    auto uniform = [](int x) __attribute__((always_inline)) { return __builtin_amdgcn_readfirstlane(x); };
    const int lo_wg = uniform(rb.lo_wg), hi_wg = uniform(rb.hi_wg), lo_w = uniform(rb.lo_w), hi_w = uniform(rb.hi_w);
    const int full_lo_w = uniform(rb.full_lo_w), full_hi_w = uniform(rb.full_hi_w);
    const bool wave_has_rows = qw0 < p.Sq;

    // ---- tile movement: one tensor's rows at a time through `st` ------------------------------------------------
    // K and V of this (batch, kv head) as raw buffers that end with the last key of the sequence: rows beyond it read as
    // zero, and so do the dims beyond head_dim (their lanes' offsets lie outside), without clamps or 64-bit addresses.
    constexpr int ES = sizeof(T);
    auto rows_of = [&](const void *base, const int64_t *st, int row_bytes) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)base + b * st[0] + g * st[1]), 0,
                                                 (key_end - 1) * row_bytes + p.D * ES, 0x00020000);
    };
    const int k_row = (int)p.ks[2] * ES, v_row = (int)p.vs[2] * ES;
    const auto k_rows = rows_of(p.k, p.ks, k_row), v_rows = rows_of(p.v, p.vs, v_row);
    const int my_row = gtid / C::LPR, my_col = gtid % C::LPR;
    auto load_rows = [&](auto &st, const auto &rows, int row_bytes, int j0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < C::NCH; i++) {
            const int col = my_col + C::LPR * (i % C::CSTEPS);
            const int at = col * 4 < p.D ? my_row * row_bytes + col * 4 * ES : (int)0x80000000;
            const int from = (j0 + C::RSTEP * (i / C::CSTEPS)) * row_bytes;
            st[i] = buffer_load4<T>(rows, at, from);
        }
    };
    auto store_rows = [&](const auto &st, int base, int pitch, int plane) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < C::NCH; i++) {
            const int at = base + (my_row + C::RSTEP * (i / C::CSTEPS)) * pitch + (my_col + C::LPR * (i % C::CSTEPS)) * 8;
            uint32_t lo[N], hi[N];
            split4<N>(st[i], lo, hi);
#pragma unroll
            for (int t = 0; t < N; t++) *LDST_PTR(uint2_t, at + t * plane) = uint2_t{lo[t], hi[t]};
        }
    };

    const int j_begin = (lo_wg / PT_BN) * PT_BN;
    const int ntiles = hi_wg > j_begin ? (hi_wg - j_begin + PT_BN - 1) / PT_BN : 0;
    float4_t st[C::NCH];  // K and V take turns
    if (ntiles > 0) load_rows(st, k_rows, k_row, j_begin + grp * PT_BN);

    // Q operand: the terms of Q[query][16 kb + 8 h2 .. +8].  The rows are read in whole lines and dealt out to the lanes
    // that own them through LDS, half of the dims at a time.
    // An f32 Q takes the scale and log2(e), so that the scores of S^T are exponents of two; 16-bit rows would need three
    // terms for that, and their scores are multiplied instead.  Where a mask is added to the scores, log2(e) waits for the
    // difference from the row's reference (see the probabilities).  Either way the largest score of a row's first tile has
    // probability 1 exactly.
    constexpr bool SCALED_Q = sizeof(T) == 4;
    bf16x8_t qt[NKB][N];
    uint32_t odd_rows = 0;  // rows that unit_in_f32 is to form
    const float score_scale = bias_on ? p.scale : p.scale * PF32_LOG2E, q_scale = SCALED_Q ? score_scale : 1.0f;
    const auto q_rows = __builtin_amdgcn_make_buffer_rsrc((void *)((const T *)p.q + b * p.qs[0] + h * p.qs[1]), 0, 0x7fffffff, 0x00020000);
    {
        constexpr int CPH = D / 8, NQ = CPH / 2;  // 16-byte pieces per half row; loads per half
        float4_t x[2][NQ], v0[C::NCH];
#pragma unroll
        for (int hf = 0; hf < 2; hf++)
#pragma unroll
            for (int i = 0; i < NQ; i++) {
                const int cid = lane + 64 * i, row = cid / CPH, dim = (cid % CPH) * 4 + hf * (D / 2);
                const int at = min(qw0 + row, p.Sq - 1) * ((int)p.qs[2] * ES) + dim * ES;
                x[hf][i] = buffer_load4<T>(q_rows, at | (dim < p.D ? 0 : (int)0x80000000), 0);
            }
        // the first V tile is requested with K and Q, so that a short call waits for memory once
        if (ntiles > 0) load_rows(v0, v_rows, v_row, j_begin + grp * PT_BN);
        const int mine = wave * C::ROWS_BYTES;
        uint32_t least = 0xffffffffu;
        float most = 0.0f;
#pragma unroll
        for (int hf = 0; hf < 2; hf++) {
            if (hf) wave_lds_sync();
#pragma unroll
            for (int i = 0; i < NQ; i++) {
                const int cid = lane + 64 * i;
                *LDST_PTR(float4_t, mine + (cid / CPH) * C::HALF_PITCH + (cid % CPH) * 16) = x[hf][i];
            }
            wave_lds_sync();
#pragma unroll
            for (int kk = 0; kk < NKB / 2; kk++) {
                uint32_t w[4][N];
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const float4_t y = *LDST_PTR(float4_t, mine + ln * C::HALF_PITCH + (16 * kk + 8 * h2 + 4 * e) * 4) * q_scale;
                    if constexpr (SCALED_Q) {
#pragma unroll
                        for (int i = 0; i < 4; i++) least = min(least, magnitude(y[i])), most = fmaxf(most, fabsf(y[i]));
                    }
                    split4<N>(y, w[2 * e], w[2 * e + 1]);
                }
#pragma unroll
                for (int i = 0; i < N; i++)
                    qt[hf * (NKB / 2) + kk][i] = __builtin_bit_cast(bf16x8_t, uint4_t{w[0][i], w[1][i], w[2][i], w[3][i]});
            }
        }
        if constexpr (SCALED_Q) {
            const uint64_t odd = __builtin_amdgcn_ballot_w64(least < magnitude(SMALLEST_IN_TERMS) || most > LARGEST_Q);
            odd_rows = (uint32_t)odd | (uint32_t)(odd >> 32);
        }
        lds_barrier();  // the tiles take the space over
        if (ntiles > 0) {
            store_rows(st, gbase, C::KP, C::K_PLANE);
            store_rows(v0, gbase + C::V_BASE, C::VP, C::V_PLANE);
        }
    }

    float16_t o[NDB];
#pragma unroll
    for (int db = 0; db < NDB; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[db][r] = 0.0f;
    // m: the row's reference (see `probability` in attn_f32.h); nmr = -m in powers of two, +inf while the row has seen no key
    float m = -INFINITY, l = 0.0f, nmr = INFINITY;
    const float log2_unit = bias_on ? PF32_LOG2E : 1.0f;
    const T *mrow = nullptr;
    if constexpr (BIAS)
        mrow = (const T *)p.mask + (int64_t)(p.mask_kind == FHIP_MASK_QK ? min(query, p.Sq - 1) : b) * p.ms0;
    // The same as a buffer.  Whole tiles read four keys per load without an address or a test per element, which cost more
    // than the tile's matrix work: f32, 8 x 512 rows, 12 heads, D = 64 with -10000 on the padding 61 -> 46 us (the scan launch below included).
    const auto mask_buf = __builtin_amdgcn_make_buffer_rsrc(
        (void *)((const T *)p.mask + (BIAS && p.mask_kind != FHIP_MASK_QK ? b * p.ms0 : 0)), 0, 0x7fffffff, 0x00020000);
    const int mask_at = (p.mask_kind == FHIP_MASK_QK ? min(query, p.Sq - 1) * (int)p.ms0 * ES : 0) + 4 * h2 * ES;

    float16_t s;
    uint32_t pt[3][8];  // the terms of the tile's probabilities, packed pairs in the operand's order
    const int k_at = gbase + ln * C::KP + h2 * 16;
    const int i16 = lane & 15, bl = (lane & 31) >> 4;
    const int v_at = gbase + C::V_BASE + (4 * h2 + (i16 >> 2)) * C::VP + (16 * bl + 4 * (i16 & 3)) * 2;

    // S^T of the tile at j0, then its probabilities: s -> pt
    auto scores = [&](int j0) __attribute__((always_inline)) {
        float bias[BIAS ? 16 : 1];
        if constexpr (BIAS) {  // requested before the matrix work that hides their latency
            if (bias_on && tl.mask_rows && j0 + PT_BN <= p.Skv) {
#pragma unroll
                for (int rq = 0; rq < 4; rq++) {
                    const float4_t x = buffer_load4<T>(mask_buf, mask_at + 8 * rq * ES, j0 * ES);
#pragma unroll
                    for (int e = 0; e < 4; e++) bias[4 * rq + e] = x[e];
                }
            } else if (bias_on) {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int key = j0 + 8 * (r >> 2) + 4 * h2 + (r & 3);
                    bias[r] = key < p.Skv ? to_float(mrow[(int64_t)key * p.ms1]) : 0.0f;
                }
            }
        }
        float16_t small;  // the sum of the products of lower terms, kept apart: fewer roundings at the size of the scores
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = small[r] = 0.0f;
        // a term's operand is read again as soon as its last product with the slice has been issued
        bf16x8_t ka[N];
        auto read_k = [&](int kb, int i) __attribute__((always_inline)) {
            ka[i] = __builtin_bit_cast(bf16x8_t, *LDST_PTR(uint4_t, k_at + i * C::K_PLANE + kb * 32));
        };
        __builtin_amdgcn_s_setprio(MATRIX_PRIO);
#pragma unroll
        for (int i = N - 1; i >= 0; i--) read_k(0, i);
#pragma unroll
        for (int kb = 0; kb < NKB; kb++)
#pragma unroll
            for (int i = N - 1; i >= 0; i--) {
#pragma unroll
                for (int j = N - 1 < 2 - i ? N - 1 : 2 - i; j >= 0; j--) {
                    if (i + j == 0) s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[i], qt[kb][j], s, 0, 0, 0);
                    else small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[i], qt[kb][j], small, 0, 0, 0);
                }
                if (kb + 1 < NKB) read_k(kb + 1, i);
            }
        // 0x100 = LDS read, 0x008 = MFMA
        __builtin_amdgcn_sched_group_barrier(0x100, N, 0);
#pragma unroll
        for (int kb = 0; kb < NKB; kb++)
#pragma unroll
            for (int i = N - 1; i >= 0; i--) {
                if (i == 0) __builtin_amdgcn_sched_group_barrier(0x008, N < 3 ? N : 3, 0);
                else if (i == 1) __builtin_amdgcn_sched_group_barrier(0x008, N < 2 ? N : 2, 0);
                else __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (kb + 1 < NKB) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
        __builtin_amdgcn_s_setprio(1 - MATRIX_PRIO);
        if constexpr (N > 1) s += small;

        // element r is key j0 + 8 (r / 4) + 4 h2 + r % 4 for query `query`
        if (!(j0 >= full_lo_w && j0 + PT_BN <= full_hi_w)) {
            asm volatile("");  // a branch: most tiles need no element test
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int key = j0 + 8 * (r >> 2) + 4 * h2 + (r & 3);
                s[r] = (key >= rb.klo && key < rb.khi) ? s[r] : -INFINITY;
            }
        }
        if constexpr (!SCALED_Q) s *= score_scale;
        if constexpr (BIAS) {
            if (bias_on) {
#pragma unroll
                for (int r = 0; r < 16; r++) s[r] += bias[r];
            }
        }
        float ts = 0.0f, pr[16];
        auto probabilities = [&](float nm) __attribute__((always_inline)) {
            float sum[2] = {0.0f, 0.0f};
#pragma unroll
            for (int r = 0; r < 16; r++) {
                pr[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], log2_unit, nm));
                sum[r & 1] += pr[r];
            }
            return sum[0] + sum[1];
        };
        ts = probabilities(nmr);
        // not at most 2^15 (NaN and +inf included): some row's reference has to move
        if (__builtin_amdgcn_ballot_w64(!(ts <= 32768.0f)) != 0) {
            float mx = s[0];
#pragma unroll
            for (int r = 1; r < 16; r++) mx = fmaxf(mx, s[r]);
            mx = half_swap_max32(mx);
            const float m_new = fmaxf(m, mx);
            const float corr = moved_reference(m, m_new, log2_unit);
            m = m_new;
            l *= corr;
#pragma unroll
            for (int db = 0; db < NDB; db++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[db][r] *= corr;
            // still no visible key: the tile's probabilities are exp2(-inf) = 0 and the row stays without a reference
            nmr = -(m * log2_unit);
            ts = probabilities(nmr == INFINITY ? 0.0f : nmr);
            if constexpr (BIAS) {
                // nothing but lowest values yet (see `probability`): those came out 0 as well, and the row comes here with every
                // tile until a score is higher
                if (bias_on) {
                    const float lowest = nmr == INFINITY && m > -INFINITY ? m : __builtin_nanf("");
                    ts = 0.0f;
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        pr[r] = s[r] == lowest ? 1.0f : pr[r];
                        ts += pr[r];
                    }
                }
            }
        }
        l += ts;
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
            uint32_t lo[3], hi[3];
            split4<3>(float4_t{pr[2 * i], pr[2 * i + 1], pr[2 * i + 2], pr[2 * i + 3]}, lo, hi);
#pragma unroll
            for (int j = 0; j < 3; j++) pt[j][i] = lo[j], pt[j][i + 1] = hi[j];
        }
    };
    // O^T += V^T . P^T: contraction slice kk holds this half-wave's keys 16 kk + 4 h2 + {0..3} and + 8
    auto pv = [&]() __attribute__((always_inline)) {
        bf16x8_t va[N];
        auto read_v = [&](int u, int i) __attribute__((always_inline)) {  // u = 2 db + kk
            const int at = v_at + (u & 1) * 16 * C::VP + (u >> 1) * 64 + i * C::V_PLANE;
            const short4_t a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDST_PTR(short4_t, at));
            const short4_t a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDST_PTR(short4_t, at + 8 * C::VP));
            const uint2_t u0 = __builtin_bit_cast(uint2_t, a0), u1 = __builtin_bit_cast(uint2_t, a1);
            va[i] = __builtin_bit_cast(bf16x8_t, uint4_t{u0[0], u0[1], u1[0], u1[1]});
        };
#pragma unroll
        for (int i = N - 1; i >= 0; i--) read_v(0, i);
#pragma unroll
        for (int db = 0; db < NDB; db++) {
            // this tile's share on its own, then one addition per tile at the size of the sum
            float16_t sum;
#pragma unroll
            for (int r = 0; r < 16; r++) sum[r] = 0.0f;
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
                const int u = 2 * db + kk;
#pragma unroll
                for (int i = N - 1; i >= 0; i--) {
#pragma unroll
                    for (int j = 2 - i; j >= 0; j--) {
                        const uint4_t w = {pt[j][4 * kk], pt[j][4 * kk + 1], pt[j][4 * kk + 2], pt[j][4 * kk + 3]};
                        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[i], __builtin_bit_cast(bf16x8_t, w), sum, 0, 0, 0);
                    }
                    if (u + 1 < 2 * NDB) read_v(u + 1, i);
                }
            }
            o[db] += sum;
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * N, 0);
#pragma unroll
        for (int u = 0; u < 2 * NDB; u++)
#pragma unroll
            for (int i = N - 1; i >= 0; i--) {
                if (i == 0) __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
                else if (i == 1) __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
                else __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (u + 1 < 2 * NDB) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            }
    };

    // Group g takes the tiles t with t % KG == g; every group runs the same number of iterations (the barriers are
    // workgroup-wide), rows beyond the last tile read as zero and are not used.
    const int niter = (ntiles + KG - 1) / KG;
    lds_barrier();
    for (int it = 0; it < niter; it++) {
        const int t = it * KG + grp;
        const int j0 = j_begin + t * PT_BN;
        const bool tile_visible = (KG == 1 || t < ntiles) && wave_has_rows && j0 < hi_w && j0 + PT_BN > lo_w;
        const bool more = it + 1 < niter;
        if (tile_visible) scores(j0);
        // V(t): every wavefront is past P.V of the group's previous tile
        if (it > 0) store_rows(st, gbase + C::V_BASE, C::VP, C::V_PLANE);
        if (more) load_rows(st, k_rows, k_row, j0 + KG * PT_BN);
        lds_barrier();
        __builtin_amdgcn_s_setprio(MATRIX_PRIO);
        if (tile_visible) pv();
        __builtin_amdgcn_s_setprio(1 - MATRIX_PRIO);
        if (more) {
            store_rows(st, gbase, C::KP, C::K_PLANE);  // the group's next K tile: every wavefront is past S^T of this one
            load_rows(st, v_rows, v_row, j0 + KG * PT_BN);
        }
        lds_barrier();
    }

    if constexpr (KG > 1) {
        // groups 1.. park (O, m, l) in LDS in 16-byte pieces per lane, group 0 folds them into its own state
        constexpr int NQ = 4 * NDB + 1, SLOT = NQ * 1024;
        static_assert((KG - 1) * U * SLOT <= KG * C::G_BYTES, "merge staging exceeds the tile buffers");
        if (grp > 0) {
            const int at = ((grp - 1) * U + wave % U) * SLOT + lane * 16;
#pragma unroll
            for (int db = 0; db < NDB; db++)
#pragma unroll
                for (int rq = 0; rq < 4; rq++)
                    *LDST_PTR(float4_t, at + (4 * db + rq) * 1024) =
                        float4_t{o[db][4 * rq], o[db][4 * rq + 1], o[db][4 * rq + 2], o[db][4 * rq + 3]};
            *LDST_PTR(float4_t, at + (NQ - 1) * 1024) = float4_t{m, l, 0.0f, 0.0f};
        }
        lds_barrier();
        if (grp > 0) return;
        float4_t ml[KG];
        float m_all = m;
#pragma unroll
        for (int src = 1; src < KG; src++) {
            ml[src] = *LDST_PTR(float4_t, ((src - 1) * U + wave) * SLOT + lane * 16 + (NQ - 1) * 1024);
            m_all = fmaxf(m_all, ml[src][0]);
        }
        const float w0 = moved_reference(m, m_all, log2_unit);
        l *= w0;
#pragma unroll
        for (int db = 0; db < NDB; db++) o[db] *= w0;
#pragma unroll
        for (int src = 1; src < KG; src++) {
            const float w = moved_reference(ml[src][0], m_all, log2_unit);
            const int at = ((src - 1) * U + wave) * SLOT + lane * 16;
            l += ml[src][1] * w;
#pragma unroll
            for (int db = 0; db < NDB; db++)
#pragma unroll
                for (int rq = 0; rq < 4; rq++) {
                    const float4_t x = *LDST_PTR(float4_t, at + (4 * db + rq) * 1024);
#pragma unroll
                    for (int e = 0; e < 4; e++) o[db][4 * rq + e] += x[e] * w;
                }
        }
        m = m_all;
    }

    // ---- out[query][dim] = O^T[dim][query] / l; with the keys split over workgroups this share's state is parked and
    // the merge kernel normalises
    const float l_tot = half_swap_sum32(l);
    // rows with a sum that is not finite (0 x inf and 0 x NaN are NaN), or with one so small that V's terms may lack bits of it
    float zero[4] = {l * 0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t least = 0xffffffffu;
#pragma unroll
    for (int db = 0; db < NDB; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            zero[r & 3] = __builtin_fmaf(o[db][r], 0.0f, zero[r & 3]);
            if constexpr (N == 3) least = min(least, magnitude(o[db][r]));
        }
    const uint64_t odd = __builtin_amdgcn_ballot_w64(!(zero[0] + zero[1] + (zero[2] + zero[3]) == 0.0f) ||
                                                     least < magnitude(l_tot * SMALLEST_IN_TERMS));
    odd_rows = wave_has_rows ? odd_rows | (uint32_t)odd | (uint32_t)(odd >> 32) : 0;
    const bool parked = nks > 1;
    float *const part = p.partials + (((int64_t)b * p.H + h) * p.Sq * nks + ksplit) * p.pf_pitch;
    const int64_t part_row = (int64_t)nks * p.pf_pitch;
    if (parked) {
        if (h2 == 0 && query < p.Sq) {
            part[query * part_row + p.D] = m;
            part[query * part_row + p.D + 1] = bias_on ? -l_tot : l_tot;  // (the sign tells the merge kernel m's unit)
        }
    } else {
        // o / l by one reciprocal and a correction of each quotient; no visible key: 0 x inf = NaN like the reference's 0 / 0
        const float inv = 1.0f / l_tot;
#pragma unroll
        for (int db = 0; db < NDB; db++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float q = o[db][r] * inv;
                o[db][r] = __builtin_fmaf(__builtin_fmaf(-q, l_tot, o[db][r]), inv, q);
            }
    }
    const int64_t ob = b * p.os[0] + h * p.os[1];
    // a wavefront's own part of LDS (with key groups: where this wavefront alone has just read)
    const int mine = KG > 1 ? wave * (4 * NDB + 1) * 1024 : wave * C::ROWS_BYTES;
    if (parked || tl.out_vec) {  // through LDS, 32 dims at a time
#pragma unroll
        for (int db = 0; db < NDB; db++) {
            wave_lds_sync();
#pragma unroll
            for (int rq = 0; rq < 4; rq++)
                *LDST_PTR(float4_t, mine + ln * C::OUT_PITCH + (8 * rq + 4 * h2) * 4) =
                    float4_t{o[db][4 * rq], o[db][4 * rq + 1], o[db][4 * rq + 2], o[db][4 * rq + 3]};
            wave_lds_sync();
            const int dim = 32 * db + (lane & 7) * 4;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = 8 * i + (lane >> 3), q = qw0 + row;
                if (q >= p.Sq || dim >= p.D) continue;
                const float4_t v = *LDST_PTR(float4_t, mine + row * C::OUT_PITCH + (lane & 7) * 16);
                if (parked) {
                    *(float4_at8_t *)(part + q * part_row + dim) = v;
                } else if (sizeof(T) == 4 || tl.out_vec == 16) {
                    *(float4_t *)((float *)p.out + ob + (int64_t)q * p.os[2] + dim) = v;
                } else if constexpr (sizeof(T) == 2) {
                    T four[4] = {from_float<T>(v[0]), from_float<T>(v[1]), from_float<T>(v[2]), from_float<T>(v[3])};
                    uint2_t w;
                    __builtin_memcpy(&w, four, 8);
                    *(uint2_t *)((T *)p.out + ob + (int64_t)q * p.os[2] + dim) = w;
                }
            }
        }
    } else if (query < p.Sq) {
#pragma unroll
        for (int db = 0; db < NDB; db++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int dim = 32 * db + 8 * (r >> 2) + 4 * h2 + (r & 3);
                if (dim < p.D) store_out<T>(p, ob + (int64_t)query * p.os[2] + dim * p.os[3], o[db][r]);
            }
    }
    if (odd_rows == 0) return;
    __threadfence();  // the stores above come first
    rb.lo_w = lo_w, rb.hi_w = hi_w, rb.full_lo_w = full_lo_w, rb.full_hi_w = full_hi_w;  // (the scalar copies)
    const RowBuffers buffers = {k_rows, v_rows, q_rows, k_row, v_row, min(query, p.Sq - 1) * ((int)p.qs[2] * ES)};
    wave_lds_sync();
    unit_in_f32<T, D>(p, lds_base + mine, buffers, bias_on ? mrow : nullptr, rb, odd_rows, lane, o, m, l);
    const float l_odd = half_swap_sum32(l);
    if (query >= p.Sq || !(odd_rows >> ln & 1)) return;
    if (parked && h2 == 0) part[query * part_row + p.D] = m, part[query * part_row + p.D + 1] = bias_on ? -l_odd : l_odd;
#pragma unroll
    for (int db = 0; db < NDB; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int dim = 32 * db + 8 * (r >> 2) + 4 * h2 + (r & 3);
            if (dim >= p.D) continue;
            if (parked) part[query * part_row + dim] = o[db][r];
            else store_out<T>(p, ob + (int64_t)query * p.os[2] + dim * p.os[3], o[db][r] / l_odd);
        }
}

// ---- which form a call takes ------------------------------------------------------------------------------------------------

static long units_of(const TermsCall &c) { return (long)c.G * ((c.Sq + 31) / 32); }

// workgroups of the form with U units each, in ns shares of the keys
static long terms_workgroups(const TermsCall &c, int U, int ns) {
    return (units_of(c) + U - 1) / U * c.B * c.Hkv * (ns > 1 ? ns : 1);
}

// The form by the numbers of its workgroups (measured on f32 calls, time per call in us; w2, w4: workgroups with 2 or 4 units):
//   (4, 1)  two workgroups per CU, least splitting per tile: grids that fill the chip twice.  Head dims above 128, one workgroup per CU
//           (106 KiB of LDS, 512 registers): a wavefront per SIMD issues its matrix and vector work in turn, 12200 cycles a tile
//           at 256, 6144 of them matrix instructions (5.3 to 5.6 us by the clock; profiles/prefill_f32_terms.txt; 16/4 heads causal, us before, on the f32 matrix instruction: 148 rows on 3510 keys
//           192 -> 80, 1024 x 1024 181 -> 119, 3191 x 3191 826 -> 555, 1500 x 6000 1577 -> 1020)
//   (4, 2)  eight wavefronts, one workgroup per CU: D = 128 1500 rows 115 against 142 for (4, 1), 4000 rows of 8 heads
//           262 against 348, 129 rows on 8003 keys (keys split over workgroups) 111 against 133
//   (2, 2)  D > 64: one wavefront per SIMD with 512 registers, half the units per workgroup, for short prompts (700 rows
//           48 against 55 for (4, 2), 200 rows 21 against 24) and others that fit the CUs once.  With the keys split there is no
//           short workgroup beside a long one unless the prompt is causal (768 rows of 8/2 heads, 288 workgroups: 33 against 36
//           with causality, 51 against 39 without; 16/4 heads, 384 workgroups: 58 against 47).  D <= 64: two workgroups per CU;
//           square causal prompts, whose later rows see more keys, are spread more evenly by half the units (1024 rows 38
//           against 47 for (4, 2), 2048 rows 111 and 2560 rows 159 against 118 and 165 for (4, 1); 3072 rows 224 against 216,
//           4096 rows 388 against 336), and up to two tiles have nothing for more than two groups (55 rows of 16/4 heads 9.4 in
//           (2, 4), 8.0)
//   (2, 4)  D <= 64, eight wavefronts: 512 rows 18 against 21.5 for (2, 2), 1000 rows of 16 heads without a mask 31
//           against 38
static TermsForm form_by_workgroups(const TermsCall &c, int ns) {
    const int cus = c.cus;
    const long w2 = terms_workgroups(c, 2, ns), w4 = terms_workgroups(c, 4, ns);
    const bool few_rows = 2L * c.Sq <= c.Skv;
    if (c.D <= 64) {
        if (c.Skv <= 2 * PT_BN) return {2, 2};
        if (2 * w2 <= (c.uneven ? 3L : 2L) * cus) return {2, 4};
        if (c.uneven && 2 * w4 <= 5L * cus) return {2, 2};
        if (!c.uneven && w4 <= cus) return {4, 2};
    } else {
        const bool fits = w2 <= cus || (ns > 1 ? c.uneven && 4 * w2 <= 5L * cus : !few_rows && 2 * w2 <= 3L * cus);
        if (fits) return {2, 2};
        if (w4 < 2L * cus) return {4, 2};
    }
    return {4, 1};
}

// Time of a call whose rows all see about the same keys, in us: rounds of workgroups that walk their tiles, and parking and
// merging the shares.  Constants fitted to 210 random calls (chunks, turns, images and encoders of 8 to 32 heads at 64 to 128
// dims, each in every form and up to 48 shares): 6 % off in the mean square.
double prefill_f32_merge_time(const TermsCall &c, int ns) {
    return 3.24 + 0.456e-6 * prefill_f32_workspace_bytes(c.B, c.Hkv * c.G, c.Sq, c.D, ns);
}
static double wide_terms_time(const TermsCall &c, int ns);
namespace {
// Of a workgroup: a tile of one of its key groups, its ends, and what a tile takes where a CU has one of two workgroups.
struct FormTimes {
    double tile, ends, alone;
    bool two_per_cu;
};
FormTimes times_of_form(int D, TermsForm f) {
    const double dims = (D <= 64 ? 64 : D <= 96 ? 96 : 128) / 64.0;
    if (f.U == 2 && f.KG == 2 && D <= 64) return {2.65, 1.4, 0.71, true};
    if (f.U == 2 && f.KG == 2) return {0.38 + 1.494 * dims, 3.9, 1.0, false};
    if (f.KG == 2) return {0.306 + 1.945 * dims, 3.45, 1.0, false};
    if (f.KG == 4) return {2.65, 3.87, 1.0, false};
    return {0.374 + 1.78 * dims, 0.8, 0.74, true};
}
}  // namespace
double prefill_f32_terms_time(const TermsCall &c, TermsForm f, int ns) {
    if (c.D > 128) return wide_terms_time(c, ns);
    const FormTimes t = times_of_form(c.D, f);
    const int chunk = ((c.Skv + ns - 1) / ns + PT_BN - 1) / PT_BN * PT_BN, n = (c.Skv + chunk - 1) / chunk;
    int tiles = chunk / PT_BN;
    // (a workgroup's rows see the window's keys and as many more as there are rows: counted for 32 rows in every form, ungrouped heads took
    // four units too often, 16 heads at 96, three sequences of 156 rows under 32 21.7 us for 13.9, over 110 chunks 1.09 of the time; wider windows
    // than 0.7 of the keys are taken for none: 32/8 heads at 128, 1100 rows under 2885 of 3984 keys would stay unsplit and take 1.21 times as long)
    const int rows = 32 * ((f.U + c.G - 1) / c.G);
    if (c.window > 0 && c.window < c.Skv && 10 * (c.window + PT_BN) < 7LL * c.Skv) tiles = std::min(tiles, ((int)c.window + rows + PT_BN - 1) / PT_BN + 1);
    const double walk = t.tile * ((tiles + f.KG - 1) / f.KG);
    const long wgs = terms_workgroups(c, f.U, n), slots = (t.two_per_cu ? 2L : 1L) * c.cus, rest = wgs % slots;
    double us = 4.9 + wgs / slots * (t.ends + walk);
    if (rest) us += t.ends + walk * (rest <= c.cus ? t.alone : 1.0);
    if (n > 1) us += prefill_f32_merge_time(c, n);
    return us;
}

// Unsplit chunks under a causal mask that need more than one round: the rows of the later rounds see the fewest keys, and start first where rows
// of few keys end.  1.15 times what the second (third) round's first workgroup takes twice (three times), or the mean load: 5 % off over nine
// chunks of 272 to 376 workgroups, which as even calls were taken for 1.1 to 1.5 times their time and split for nothing (us, four sequences
// of 1071 rows of 8/4 heads at 128 on 2216 keys 203 unsplit and 261 in two shares, three of 1832 of 8/2 at 96 on 3665 289 and 336).
double prefill_f32_unsplit_time(const TermsCall &c, TermsForm f) {
    const double even = prefill_f32_terms_time(c, f, 1);
    if (c.D > 128 || !c.causal || c.window > 0) return even;
    const FormTimes t = times_of_form(c.D, f);
    const double walk = t.tile * (((c.Skv + PT_BN - 1) / PT_BN + f.KG - 1) / f.KG), part = (double)c.Sq / c.Skv;
    const double wgs = (double)terms_workgroups(c, f.U, 1), slots = (t.two_per_cu ? 2.0 : 1.0) * c.cus;
    if (wgs <= slots) return even;
    double us = std::max(t.ends + walk, 1.08 * wgs / slots * (t.ends + walk * (1.0 - 0.5 * part)));
    us = std::max(us, 2.0 * (t.ends + walk * (1.0 - part * slots / wgs)));
    if (wgs > 2 * slots) us = std::max(us, 3.0 * (t.ends + walk * (1.0 - part * 2.0 * slots / wgs)));
    return std::min(even, 4.9 + 1.15 * us);
}

// The same above head_dim 128, where the form is (4, 1) with one workgroup per CU, of uneven calls too: even shares in rounds; of uneven
// ones, dealt out the longest first, the longest, the mean load, or twice (three times) the first workgroup of the second (third) round.
// Over 420 random calls at 160 to 256 dims in up to 48 shares it is 6 % off in the mean square, 9 % under a window.
// Under a window a row block sees the window's keys and meets few of the shares; the
// workgroups of the others still split Q, park a state and have it merged (us, planned without the window and with it: 16/8 heads at 256,
// 786 rows under a window of 127 59 -> 47; 12/12 at 160, 1317 under 103 58 -> 46; 6/3 at 192, three sequences of 718 under 117 50 -> 38).
static double wide_terms_time(const TermsCall &c, int ns) {
    const double tile = 1.33 * (c.D <= 192 ? 3 : 4), ends = 6.9;
    const int chunk = ((c.Skv + ns - 1) / ns + PT_BN - 1) / PT_BN * PT_BN, n = (c.Skv + chunk - 1) / chunk;
    const long wgs = terms_workgroups(c, 4, 1);
    const int rows = std::min(c.Sq, 32 * ((4 + c.G - 1) / c.G));  // of a workgroup
    const bool narrow = c.window > 0 && c.window < c.Skv - rows;
    const double sight = narrow ? (double)c.window + rows : c.Skv;  // keys from the first to the last that a workgroup's rows see
    double most = chunk / PT_BN;
    if (narrow && sight <= chunk) most = (int)(sight - 1 + PT_BN - 1) / PT_BN + 1;
    const double longest = ends + tile * most;
    double us;
    if (!c.uneven) {
        us = (double)((wgs * n + c.cus - 1) / c.cus) * longest;
    } else {
        const double first = c.Skv > c.Sq ? c.Skv - c.Sq : 0.0;  // keys before the first row
        // workgroups that see this many keys of their share
        auto with_keys = [&](double keys) {
            double sum = 0.0;
            for (int i = 0; i < n; i++) {
                const double from = std::max(first, (double)i * chunk + keys);
                const double to = narrow ? std::min<double>(c.Skv, std::min<double>(c.Skv, (i + 1.0) * chunk) + sight - keys) : c.Skv;
                const double part = (to - from) / (c.Skv - first);
                sum += part < 0.0 ? 0.0 : part > 1.0 ? 1.0 : part;
            }
            return sum * wgs;
        };
        auto time_of = [&](double nth) {  // of the nth workgroup
            if (with_keys(0.0) < nth) return narrow && wgs * n >= nth ? ends : 0.0;
            double keys = 0.0;
            for (double step = 0.5 * chunk; step >= 16.0; step *= 0.5)
                if (keys + step <= sight && with_keys(keys + step) >= nth) keys += step;
            return ends + tile / PT_BN * keys;
        };
        double seen = (first + c.Skv) * 0.5;  // by a row in the mean
        if (narrow) seen = first >= sight ? sight : (0.5 * (sight * sight - first * first) + sight * (c.Skv - sight)) / (c.Skv - first);
        const double load = wgs * (n * ends + seen / PT_BN * tile) / c.cus;
        us = std::max({longest, 1.08 * load, 2.0 * time_of(c.cus + 1.0), 3.0 * time_of(2.0 * c.cus + 1.0)});
    }
    us += 4.9;
    if (n > 1) us += prefill_f32_merge_time(c, n);
    return us;
}

TermsForm prefill_f32_terms_quickest(const TermsCall &c, int ns) {
    if (c.D > 128 || !c.f32) return {4, 1};
    TermsForm best = {4, 1};
    double least = prefill_f32_terms_time(c, best, ns);
    for (const TermsForm f : {TermsForm{4, 2}, TermsForm{2, 2}, TermsForm{2, 4}}) {
        if (f.KG == 4 && c.D > 64) continue;
        const double us = prefill_f32_terms_time(c, f, ns);
        if (us < least) least = us, best = f;
    }
    return best;
}

// Where all rows see about the same keys the rule above leaves much to gain, and the form is the quickest by the time above if that
// is 10 % better (us a call: 16 heads without a mask, 1356 rows at 128 169 -> 99; 6 encoder sequences of 436 tokens 41.5 -> 30.6, 11
// of 169 23.2 -> 18.4; at 7 % ten sequences of 154, 240 workgroups of five tiles, 16.4 -> 17.1).  Up to 128 rows the rule is as good.
TermsForm prefill_f32_terms_form(const TermsCall &c, int ns) {
    if (c.D > 128 || !c.f32) return {4, 1};
    const TermsForm ordinary = form_by_workgroups(c, ns);
    if (c.uneven || c.Sq <= 128 || c.Skv <= 2 * PT_BN) return ordinary;
    const TermsForm other = prefill_f32_terms_quickest(c, ns);
    return prefill_f32_terms_time(c, other, ns) < 0.9 * prefill_f32_terms_time(c, ordinary, ns) ? other : ordinary;
}

// (of f32 tensors)
TermsCall prefill_f32_terms_call(const AttnParams &p) {
    const bool uneven = prefill_f32_uneven(p.Sq, p.Skv, p.D, p.analytic && p.causal, p.mask_kind == FHIP_MASK_QK, p.q_pos_offset, p.window);
    return {p.B, p.Hkv, p.G, p.Sq, p.Skv, p.D, p.cus > 0 ? p.cus : 256, uneven, p.analytic ? p.window : 0, true,
            (p.analytic && p.causal) || p.mask_kind == FHIP_MASK_QK};
}

template <typename T, int U, int KG, int MODE>
static int launch_form(const AttnParams &p_in, hipStream_t stream) {
    AttnParams p = p_in;
    const int cus = p.cus > 0 ? p.cus : 256;
    const long blocks = terms_workgroups(prefill_f32_terms_call(p), U, p.pf_nsplit);
    if (blocks > 0x7fffffffL) {
        set_error("prefill f32: too many workgroups (%ld)", blocks);
        return FHIP_ERR_UNSUPPORTED;
    }
    TermsLaunch tl;
    const unsigned nks = p.pf_nsplit > 1 ? p.pf_nsplit : 1, groups = (unsigned)(p.B * p.Hkv), nwg = (unsigned)(blocks / nks / groups);
    tl.level_pitch = 0;
    // (grids of one round too: without it calls of 500 rows take 2 to 5 % longer, those of 300 1 to 2 % less; under a window the same
    // workgroups of a share still see alike: the grid's order takes 1.07 to 1.16 times as long in two to eight shares of 120 random prompts)
    if (p.D > 128 && nks > 1 && prefill_f32_terms_call(p).uneven) tl.level_pitch = std::max(1, (int)((int64_t)p.pf_chunk * p.G / (32 * U)));
    tl.g_magic = p.G > 1 ? (uint32_t)((0x100000000ull + p.G - 1) / p.G) : 0;
    const bool two_per_cu = (KG == 1 && p.D <= 128) || (U * KG == 4 && p.D <= 64);
    tl.snake = (two_per_cu && blocks > cus && blocks <= 2L * cus) ? (int)((cus + nks * groups - 1) / (nks * groups)) : 0;
    // rows of the result written in 16-byte (f32) or 8-byte pieces
    const int oeb = sizeof(T) == 4 || p.out_f32 ? 4 : 2;
    tl.out_vec = p.os[3] == 1 && (uintptr_t)p.out % (4 * oeb) == 0 ? 4 * oeb : 0;
    for (int i = 0; i < 3; i++)
        if (p.os[i] % 4 != 0) tl.out_vec = 0;
    // rows of the mask in 16-byte (f32, element-aligned) or 8-byte pieces, within a buffer's 32-bit offsets
    const int64_t mask_span = ((p.mask_kind == FHIP_MASK_QK ? (int64_t)(p.Sq - 1) * p.ms0 : 0) + p.Skv) * (int64_t)sizeof(T);
    tl.mask_rows = p.mask_kind != FHIP_MASK_NONE && p.ms1 == 1 && p.ms0 >= 0 && mask_span < 0x7fffffffLL &&
                   (sizeof(T) == 4 || ((uintptr_t)p.mask % 8 == 0 && p.ms0 % 4 == 0));
    dim3 grid(nks, groups, nwg), block(64 * U * KG);
    switch ((p.D + 31) / 32 * 32) {  // the kernel's D is head_dim rounded up to a multiple of 32
        case 32: FHIP_LAUNCH_MAIN((prefill_f32_terms_kernel<T, 32, U, KG, MODE>), grid, block, stream, p, p, tl); break;
        case 64: FHIP_LAUNCH_MAIN((prefill_f32_terms_kernel<T, 64, U, KG, MODE>), grid, block, stream, p, p, tl); break;
        case 96:
            if constexpr (MODE != PF32_EITHER && KG < 4) FHIP_LAUNCH_MAIN((prefill_f32_terms_kernel<T, 96, U, KG, MODE>), grid, block, stream, p, p, tl);
            break;
        case 128:
            if constexpr (MODE != PF32_EITHER && KG < 4) FHIP_LAUNCH_MAIN((prefill_f32_terms_kernel<T, 128, U, KG, MODE>), grid, block, stream, p, p, tl);
            break;
        case 160:
        case 192:
            if constexpr (sizeof(T) == 4 && U == 4 && KG == 1 && MODE == PF32_INTERVALS) FHIP_LAUNCH_MAIN((prefill_f32_terms_kernel<T, 192, U, KG, MODE>), grid, block, stream, p, p, tl);
            break;
        case 224:
        case 256:
            if constexpr (sizeof(T) == 4 && U == 4 && KG == 1 && MODE == PF32_INTERVALS) FHIP_LAUNCH_MAIN((prefill_f32_terms_kernel<T, 256, U, KG, MODE>), grid, block, stream, p, p, tl);
            break;
        default: set_error("prefill f32 kernel: head_dim %d is not a multiple of 4 up to 256", p.D); return FHIP_ERR_UNSUPPORTED;
    }
    FHIP_HIP_CHECK(hipGetLastError());
    return FHIP_OK;
}

template <typename T, int MODE>
static int launch_terms(const AttnParams &p, hipStream_t stream) {
    // 16-bit storage takes (4, 1) always
    if constexpr (sizeof(T) == 4) {
        const TermsForm f = prefill_f32_terms_form(prefill_f32_terms_call(p), p.pf_nsplit > 1 ? p.pf_nsplit : 1);
        if (f.U == 2 && f.KG == 4) return launch_form<T, 2, 4, MODE>(p, stream);
        if (f.U == 2) return launch_form<T, 2, 2, MODE>(p, stream);
        if (f.KG == 2) return launch_form<T, 4, 2, MODE>(p, stream);
    }
    return launch_form<T, 4, 1, MODE>(p, stream);
}

// (16-bit storage above head_dim 128 is not asked for: attn_prefill_mfma_wide.hip has it.)
// K and V rows are fetched through 32-bit buffer offsets: rows must not overlap, and one (batch, kv head) slice must span
// less than 2 GiB, the tiles behind its end included.
bool prefill_f32_terms_takes(const AttnParams &p) {
    const int64_t rows = (int64_t)p.Skv + 8 * PT_BN, units = (int64_t)p.G * ((p.Sq + 31) / 32);
    // (grid dimensions, and the exactness of unit / G by multiplication)
    if ((int64_t)p.B * p.Hkv > 65535 || units > 65535 || units * p.G > 0x7fffffffLL) return false;
    if (p.qs[2] < 0 || (int64_t)p.Sq * p.qs[2] * 4 >= 0x7fffffffLL) return false;
    return p.D <= 256 && p.ks[2] >= p.D && p.vs[2] >= p.D && rows * p.ks[2] * 4 < 0x7fffffffLL && rows * p.vs[2] * 4 < 0x7fffffffLL;
}

// A BatchKeyMask whose row every wavefront can look at for itself, four keys per load and all loads at once: no scan launch.
// Longer rows, rows of a QKMask (each read by all heads) and 16-bit rows, whose last piece a buffer's bounds would cut, are
// scanned once per call.
bool prefill_f32_terms_scans(const AttnParams &p, fhip_dtype dtype) {
    return dtype == FHIP_F32 && p.mask_kind == FHIP_MASK_BATCH_KEY && p.D <= 64 && p.Skv <= SCAN_KEYS && p.ms1 == 1 &&
           prefill_f32_terms_takes(p);
}

int launch_prefill_f32_terms(const AttnParams &p, fhip_dtype dtype, int mode, hipStream_t stream) {
    auto by_type = [&](auto type) {
        typedef decltype(type) T;
        if (mode == PF32_EITHER) return launch_terms<T, PF32_EITHER>(p, stream);
        if (mode == PF32_BIAS) return launch_terms<T, PF32_BIAS>(p, stream);
        return launch_terms<T, PF32_INTERVALS>(p, stream);
    };
    if (dtype == FHIP_F16) return by_type(half_t{});
    if (dtype == FHIP_BF16) return by_type(bf16_t{});
    return by_type(float{});
}

}  // namespace fhip
