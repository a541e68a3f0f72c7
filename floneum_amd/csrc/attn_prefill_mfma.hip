// Prefill attention for f16 / bf16 on the gfx950 matrix cores.
//
// Workgroup = 8 wavefronts = 256 query rows of one (batch, head); each wavefront owns 32 rows.
// Keys/values are walked in tiles of 64 rows that go from global memory straight into a four-stage
// LDS ring (direct-to-LDS buffer loads, no staging registers).  Per tile and wavefront:
//   S^T (64 keys x 32 queries)  = K_tile . Q^T      v_mfma_f32_32x32x16  (A = K from LDS, B = Q in registers)
//   scale * log2(e) (rr) multiplies the scores in f32: a probability is exp2(fma(s, rr, -m * rr)), one fused
//   multiply-add and one exponential per score, with m the row's reference exponent
//   online softmax down the key axis: with S^T every lane owns ONE query column and 16 keys of it per 32-key
//   block, so row sums are in-lane folds (the two half-rows are added once, at the end).  No maximum is taken
//   per tile: the reference m is the maximum the row had when it was last set, and it is moved (and l and O
//   rescaled) only when a lane's probabilities of a tile sum to more than 2^15, i.e. before one of them could
//   leave the 16-bit type's range; on random data that is the first tile and almost never again
//   O^T (D x 32 queries)       += V_tile^T . P^T    A = V^T read from row-major LDS with the
//   transposing LDS load ds_read_b64_tr_b16, B = P^T taken straight from the S^T accumulator
//   registers (the contraction index is permuted identically on both operands)
// The two wavefronts that share a SIMD (w and w + 4) run half a tile out of phase: while one is in
// its matrix phase (S^T of the current tile, P.V of the previous one, tile loads) the other is in its
// vector phase (softmax), so the MFMA pipe and the VALU are busy at the same time.
// Phases are separated by workgroup barriers; the tile loads ride on the same barriers.  The vector
// phase uses no dot-product instructions: on this chip they queue behind the MFMAs of the other
// wavefront instead of running beside them.
// Bound: power at head_dim 128 (4096 x 4096 keys, 16 heads, no mask, f16: 121 us = 1.13 PFLOP/s); below, a vector phase
// takes as long as a matrix phase or longer: its 111 vector instructions take a lone wavefront 617 cycles and beside the
// matrix instructions of the other 785, the 16 / 22 / 24 matrix instructions of head_dim 64 / 80 / 96 take 512 / 704 / 768.
// So everything but the softmax itself is done in the matrix phase, in the shadow of its instructions: tile loads, addresses,
// the mask test (an instruction on the scalar unit costs a lone wavefront as much as one on the vector unit).  f16, the
// call above at head_dim 64 / 80 / 96: 88 -> 74, 100 -> 90, 107 -> 97 us (loads, their addresses and an LDS wait in the
// vector phase before: 1350 cycles, now about 950); causal, 32/8 heads, 4000 rows at 64: 97 -> 80.
// All accumulation is f32; P is rounded to the input type for the second product.
// Key-split form (template parameter KS): the workgroup owns 128 query rows and its two wavefront groups
// take alternate key tiles of the same rows, each through the same matrix / vector phases, and merge their
// (m, l, O) through LDS at the end: twice the workgroups, half the longest one, for grids that do not fill
// the chip (see prefill_mfma_block_rows).
// Masking is by interval: every query row sees one range of keys, known analytically (causal with
// offset, sliding window, per-batch kv length, tail of the key axis) or read from the interval form
// of a dense mask tensor (attn_bounds.h, mask_intervals.hip); key tiles that are invisible to the
// whole workgroup are never loaded, and tiles fully visible to a wavefront skip the per-element test.
//
// Reference semantics: fusor-ml/fusor/src/composite/flash_attention.rs:141-199, f32 accumulation
// of 16-bit inputs as fusor-ml/core/src/composite/flash_attention.rs:186-203,323-327; head
// mapping kv_head = head / (H / Hkv) (core :135-137,163-167).
#include <algorithm>
#include <type_traits>

#include "attn_bounds.h"
#include "common.h"
#include "device_utils.h"

namespace fhip {

constexpr int PF_WAVES = 8;
constexpr int PF_BM = 32 * PF_WAVES;  // query rows per workgroup
constexpr int PF_BN = 64;             // key rows per tile
constexpr float PF_LOG2E = 1.4426950408889634f;

#define LDS_PTR(type, byte_off) ((__attribute__((address_space(3))) type *)(lds_base + (byte_off)))

template <typename T>
struct Mma;
template <>
struct Mma<half_t> {
    typedef half8_t vec8;
    static __device__ __forceinline__ float16_t mfma(vec8 a, vec8 b, float16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float x, float y) {
        half2_t h = {(half_t)x, (half_t)y};
        return __builtin_bit_cast(uint32_t, h);
    }
};
template <>
struct Mma<bf16_t> {
    typedef bf16x8_t vec8;
    static __device__ __forceinline__ float16_t mfma(vec8 a, vec8 b, float16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float x, float y) {
        typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
        const bf16x2_t h = {(__bf16)x, (__bf16)y};  // v_cvt_pk_bf16_f32: round to nearest even
        return __builtin_bit_cast(uint32_t, h);
    }
    static __device__ __forceinline__ vec8 scaled(vec8 q, float c) {
#pragma unroll
        for (int e = 0; e < 8; e++) q[e] = (__bf16)((float)q[e] * c);
        return q;
    }
};

// LDS image of a 64-row tile.  Rows are kept in NG groups: row r sits in group r % NG at position r / NG.  A group is what
// one wavefront-wide direct-to-LDS load writes (D = 128: 4 rows, D = 64: 8), or three of them (D = 96: 16 rows), whole
// kilobytes either way, so that every lane of every load moves 16 bytes.  Groups are padded apart so that
//   - rows r .. r + 3 at one column fall 16 bytes apart modulo the 256-byte bank period, and the sixteen rows that the LDS
//     serves at once in a 128-bit read (four such runs) fall into sixteen different places  (K: pitch of a group + 16)
//   - the 4 rows x 64 bytes a half-wavefront reads with the transposing load fall 64 bytes apart  (V: pitch + 64)
template <int D, bool KS>
struct PfCfg {
    static constexpr int ROWB = D * 2;                               // bytes per tile row
    static constexpr int NG = D == 128 ? 16 : D == 96 ? 4 : 8;       // groups of a tile
    static constexpr int KG = PF_BN / NG * ROWB + 16;                // K group pitch, bytes
    static constexpr int VG = PF_BN / NG * ROWB + 64;                // V group pitch, bytes
    static constexpr int K_BYTES = NG * KG;
    static constexpr int V_BYTES = NG * VG;
    static constexpr int CPR = D / 8;                                // 16-byte chunks per row
    static constexpr int LOADS = PF_BN * ROWB / 4096;                // loads of each of the four wavefronts that move a tile
    static constexpr int OFFSETS = NG == 4 ? LOADS : 1;              // (their lanes' offsets differ by a uniform value otherwise)
    // tile buffers.  Unsplit form: four stages of (K tile, V tile), tile t in stage t % 4.  Key-split form
    // (KS): a ring of five K tiles followed by a ring of four V tiles (see the slot schedule in the kernel).
    static constexpr int STAGE = K_BYTES + V_BYTES;
    static constexpr int NK = KS ? 5 : 4, NV = 4;
    static constexpr int LDS_BYTES = KS ? NK * K_BYTES + NV * V_BYTES : 4 * STAGE;
    static constexpr int BM = KS ? PF_BM / 2 : PF_BM;                // query rows per workgroup
};

__device__ __forceinline__ float half_swap_max(float x) {
    // max of x with the value held by the lane 32 away
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_swap_sum(float x) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// D: head_dim rounded up to 64, 96 or 128, the width of the tiles and of O.  QD: the dims contracted in K . Q^T, head_dim
// rounded up to 16.  PAD: head_dim is less than D; the dims behind it are zero in Q, K and V (their lanes fetch from beyond
// the buffer) and are not written.
template <typename T, int D, int QD, bool PAD, bool KS>
__global__ __launch_bounds__(64 * PF_WAVES, 2) void prefill_mfma_kernel(AttnParams p, int nqb, int out_vec) {
    request_arguments<AttnParams, int, int>();
    typedef PfCfg<D, KS> C;
    typedef typename Mma<T>::vec8 vec8;
    constexpr int STAGE = C::STAGE;
    constexpr int BM = C::BM;
    __shared__ __attribute__((aligned(16))) char smem[C::LDS_BYTES];
    auto lds_base = (__attribute__((address_space(3))) char *)smem;

    if (p.iv_bad && *p.iv_bad == p.bad_tag) return;  // the mask is not made of intervals: the general kernel takes the call
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // scalar: everything derived from it is uniform
    const int lane = tid & 63;
    const int ln = lane & 31;      // query column / key row owned inside a 32-wide MFMA block
    const int h2 = lane >> 5;      // which half of the contraction slice
    const int group = wave >> 2;   // wavefronts w and w + 4 share a SIMD and run out of phase

    // workgroup -> (query block, batch, head): long query blocks first, and heads laid out so
    // the workgroups that land on one XCD (id % 8) share a KV head whenever H is a multiple of 8
    // Packed form (key-split form only, at most 32 query rows, GQA group a multiple of 4): the workgroup's four row
    // blocks are rows 0..31 of four query heads that share a KV head, so the K and V tiles it moves serve all four
    // and a few new rows on a long cache read the cache once per KV head, not once per query head.
    const int pack = KS ? p.pf_pack : 0;
    const int heads = pack ? p.H / 4 : p.H;  // head units per batch entry
    const int bh_count = p.B * heads;
    const int nks = max(p.pf_nsplit, 1);
    const int ksplit = blockIdx.x % nks;  // which share of the keys (0 when the keys are not split over workgroups)
    const int id = blockIdx.x / nks;
    const int qb = nqb - 1 - id / bh_count;
    int rem = id % bh_count;
    const int b = rem / heads;
    int h = rem % heads;
    if (pack) h = 4 * h + (wave & 3);
    else if ((p.H & 7) == 0) h = (h & 7) * (p.H >> 3) + (h >> 3);
    const int g = h / p.G;
    // Rows of a tile beyond the sequence's own keys (kv_lens below the view's length: a ragged batch in one cache
    // allocation) read as zero (the buffers end there): what such rows hold, NaN included, must not reach the result as 0 x NaN in P . V.
    // (likewise the rows behind the last query's own position when the call says where its rows stand inside a longer
    // cache view: a causal descriptor with q_pos_offset + Sq below the view's length)
    int key_end = p.kv_lens ? min(p.Skv, max(p.kv_lens[b], 1)) : p.Skv;
    if (p.analytic && p.causal) key_end = (int)min((int64_t)key_end, max(p.q_pos_offset + p.Sq, (int64_t)1));

    const int q0 = pack ? 0 : qb * BM;
    const int qw0 = pack ? 0 : q0 + 32 * (KS ? (wave & 3) : wave);  // KS: both groups own the same 128 rows
    const int query = qw0 + ln;
    RowBounds rb = row_bounds(p, b, q0, pack ? 32 : BM, qw0, lane);
    if (nks > 1) {  // few query rows on a long cache: this workgroup takes one share of the keys
        const int c_lo = ksplit * p.pf_chunk, c_hi = c_lo + p.pf_chunk;
        rb.lo_wg = max(rb.lo_wg, c_lo), rb.hi_wg = min(rb.hi_wg, c_hi);
        rb.lo_w = max(rb.lo_w, c_lo), rb.hi_w = min(rb.hi_w, c_hi);
        rb.full_lo_w = max(rb.full_lo_w, c_lo), rb.full_hi_w = min(rb.full_hi_w, c_hi);
        rb.klo = max(rb.klo, c_lo), rb.khi = min(rb.khi, c_hi);
    }
    const int lo_wg = rb.lo_wg, hi_wg = rb.hi_wg, lo_w = rb.lo_w, hi_w = rb.hi_w;
    const int full_lo_w = rb.full_lo_w, full_hi_w = rb.full_hi_w, klo = rb.klo, khi = rb.khi;
    const int qrow = min(query, p.Sq - 1);
    const int hd = PAD ? p.D : D;  // the head dim itself
    const bool wave_has_rows = qw0 < p.Sq;

    // Q^T operand: Q[query][16 kb + 8 h2 .. +8], kept in registers for the whole kernel
    // (the loads are issued here; whatever scaling they take waits until the first K/V tiles are on their way too)
    const float scale2 = p.scale * PF_LOG2E;
    // rr multiplies every score in f32 right before exp2: the scores are then the f32 dot product times the scale, one
    // rounding, as the reference computes them (fusor-ml/fusor/src/composite/flash_attention.rs:145).  Folding scale2 into
    // Q instead would save that multiply but round Q's elements a second time (11 bits in f16, 8 in bf16), an error that
    // grows in proportion to the scores.  The S^T accumulators and m are in units of 1 / rr.
    // bf16 at the kernel's own head dims: Q takes the power of two in scale2 (pw), which is exact down to bf16's smallest
    // normal value and keeps dot products of very large elements inside f32's range.  f16 takes none of it: elements below
    // 2^-14 / pw would become subnormal and lose bits, and the products of f16 elements cannot leave f32's range.
    constexpr bool FOLD = std::is_same<T, bf16_t>::value && !PAD;
    const float pw = FOLD ? __uint_as_float(__float_as_uint(scale2) & 0x7F800000u) : 1.0f;
    const float rr = FOLD ? scale2 / pw : scale2;
    vec8 qreg[QD / 16];
    {
        const uint16_t *qp = (const uint16_t *)p.q + b * p.qs[0] + h * p.qs[1] + (int64_t)qrow * p.qs[2];
#pragma unroll
        for (int kb = 0; kb < QD / 16; kb++) {
            uint4_t raw = {0, 0, 0, 0};
            if (!PAD || 16 * kb + 8 * h2 < hd) raw = *(const uint4_t *)(qp + 16 * kb + 8 * h2);
            qreg[kb] = __builtin_bit_cast(vec8, raw);
        }
    }

    const int j_begin = (lo_wg / PF_BN) * PF_BN;
    const int ntiles = hi_wg > j_begin ? (hi_wg - j_begin + PF_BN - 1) / PF_BN : 0;

    // K and V of this (batch, kv head) as raw buffers: a row beyond the end of the key axis reads as
    // zero, so the tile loop needs neither clamps nor 64-bit address arithmetic
    const uint16_t *kg = (const uint16_t *)p.k + b * p.ks[0] + g * p.ks[1];
    const uint16_t *vg = (const uint16_t *)p.v + b * p.vs[0] + g * p.vs[1];
    const int krow_bytes = (int)p.ks[2] * 2, vrow_bytes = (int)p.vs[2] * 2;

    float16_t o[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[db][r] = 0.0f;
    // m: the row's reference exponent, in units of the S^T accumulators (1 / rr of a base-2 exponent): probabilities are
    // exp2((s - m) * rr), formed as exp2(fma(s, rr, nmr)) with nmr = -m * rr.  While the row has seen no key m is -inf and
    // nmr +inf, which sends the first tile with a visible key through the branch that sets m (see softmax below).
    float m = -INFINITY, l = 0.0f, nmr = INFINITY;
    float16_t zero16;
#pragma unroll
    for (int r = 0; r < 16; r++) zero16[r] = 0.0f;

    using std::integral_constant;
    // ---- tile movement: global -> LDS directly (no registers) --------------------------------------
    // The four wavefronts of a group move one whole tile with LOADS loads each.  Load j of wavefront w writes LDS group
    // w + 4 j (D = 96: the j-th kilobyte of group w); its lanes fetch that group's 16-byte chunks in order (which is how
    // the hardware lays out a direct load).
    // Unsplit form: group 1 moves the K tiles, group 0 the V tiles.  Key-split form: the group that is in
    // its vector phase moves one K and one V tile.
    // The tensors as raw buffer descriptors (base, no stride, size in bytes, 32-bit raw format): a row beyond
    // the end of the key axis reads as zero.
    const bool moves_k = group == 1;
    const int wv = wave & 3;
    auto descriptor = [&](const uint16_t *base, int row_bytes) __attribute__((always_inline)) {
        const uint64_t ptr = (uint64_t)base;
        return uint4_t{(uint32_t)ptr, (uint32_t)(ptr >> 32) & 0xffffu, (uint32_t)((key_end - 1) * row_bytes + hd * 2),
                       0x00020000u};
    };
    const uint4_t krs = descriptor(kg, krow_bytes), vrs = descriptor(vg, vrow_bytes);
    int gofs_k[C::OFFSETS], gofs_v[C::OFFSETS];
#pragma unroll
    for (int j = 0; j < C::OFFSETS; j++) {
        const int chunk = lane + 64 * j, row = C::NG * (chunk / C::CPR) + wv, col = chunk % C::CPR;
        const bool padding = PAD && col * 8 >= hd;
        gofs_k[j] = padding ? 0x7ffffff0 : row * krow_bytes + col * 16;
        gofs_v[j] = padding ? 0x7ffffff0 : row * vrow_bytes + col * 16;
    }
    // where tile t lives in LDS
    auto k_stage = [&](int t) __attribute__((always_inline)) { return KS ? (int)((uint32_t)t % C::NK) * C::K_BYTES : (t & 3) * STAGE; };
    auto v_stage = [&](int t) __attribute__((always_inline)) {
        return KS ? C::NK * C::K_BYTES + (t & 3) * C::V_BYTES : (t & 3) * STAGE + C::K_BYTES;
    };
    // a tile that starts beyond the key axis is never used: clamp the (uniform) offset so it stays
    // inside 32 bits; rows past Skv inside a used tile are out of range of the buffer and read 0
    // (uniform values, pinned to scalar registers, which is what the instruction takes.  M0 takes an LDS address, not an
    // offset into the tile buffers: they are the kernel's only LDS variable and start at 0, which the compiler folds in.
    // Written as assembly on purpose: the compiler would otherwise make every later LDS read of this wavefront wait for
    // these loads, whose data is not due before a later barrier.)
    auto issue = [&](const uint4_t rs, const int (&gofs)[C::OFFSETS], int row_bytes, int soff, int lbase, int pitch, int j)
                     __attribute__((always_inline)) {
        const int lds = lbase + (C::NG == 4 ? 1024 * j : 4 * j * pitch), from = soff + (C::NG == 4 ? 0 : 4 * j * row_bytes);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     :
                     : "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(gofs[C::OFFSETS > 1 ? j : 0]), "s"(rs),
                       "s"(__builtin_amdgcn_readfirstlane(from))
                     : "m0");
    };
    auto row_offset = [&](int tile, int row_bytes) __attribute__((always_inline)) { return min(j_begin + tile * PF_BN, p.Skv) * row_bytes; };
    const int lds0 = (int)(uint32_t)(uintptr_t)lds_base;
    auto issue_k = [&](int tile, int j) __attribute__((always_inline)) {
        issue(krs, gofs_k, krow_bytes, row_offset(tile, krow_bytes), lds0 + k_stage(tile) + wv * C::KG, C::KG, j);
    };
    auto issue_v = [&](int tile, int j) __attribute__((always_inline)) {
        issue(vrs, gofs_v, vrow_bytes, row_offset(tile, vrow_bytes), lds0 + v_stage(tile) + wv * C::VG, C::VG, j);
    };
    // Load n of those that a matrix phase issues.  Unsplit form: of one tile of this group's tensor (K: group 1, V: group 0).
    // Key-split form, slot s: of K(s + 4) and V(s + 1).
    constexpr int PHASE_LOADS = KS ? 2 * C::LOADS : C::LOADS;
    const uint4_t mrs = moves_k ? krs : vrs;
    const int mrow_bytes = moves_k ? krow_bytes : vrow_bytes, mpitch = moves_k ? C::KG : C::VG;
    const int mbase = lds0 + (moves_k ? 0 : C::K_BYTES) + wv * mpitch;
    int mgofs[C::OFFSETS];
#pragma unroll
    for (int j = 0; j < C::OFFSETS; j++) mgofs[j] = moves_k ? gofs_k[j] : gofs_v[j];
    auto load = [&](int at, int n) __attribute__((always_inline)) {
        if (n >= PHASE_LOADS) return;
        if constexpr (KS) {
            if (n & 1) issue_v(at + 1, n >> 1);
            else issue_k(at + 4, n >> 1);
        } else {
            issue(mrs, mgofs, mrow_bytes, row_offset(at, mrow_bytes), mbase + (at & 3) * STAGE, mpitch, n);
        }
    };
    auto load_all = [&](int at) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < PHASE_LOADS; n++) load(at, n);
    };
    // all but the most recent N loads of this wavefront have landed
    auto wait_loads = [&](auto n) __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"i"(decltype(n)::value) : "memory");
    };
    // local tile index -> tile: in the key-split form group g owns the tiles t with t % 2 == g
    auto tile_of = [&](int i) __attribute__((always_inline)) { return KS ? 2 * i + group : i; };

    float16_t s[2];     // S^T of the tile in flight
    uint32_t pk[2][8];  // its probabilities, packed pairs in the MFMA operand order

    // A matrix phase: S^T of tile i (QK) and P.V of tile i - 1 (PV), and the tile loads of the slot.  S^T's K operands of the
    // first PRE contraction slices have been read in the vector phase before (PREFETCHED), the others leave the LDS several
    // matrix instructions ahead of their use, and V's likewise; each step is fenced, so that neither the reads nor the
    // loads gather in front of the matrix instructions.
    // O^T += V^T . P^T: contraction slice (t, kk) holds this half-wave's keys 32 t + 16 kk + 4 h2 + {0..3} and + 8
    constexpr int NDB = D / 32, NKB = QD / 16;
    constexpr int PFK = (D == 128) ? 2 : 4;  // K operand slices in flight (register budget)
    // Contraction slices read in the vector phase.  None where that phase is much the longer one: head_dim 64, 4096 x 4096 keys
    // 76.8 -> 75.4 us; at 80 and 96 no difference, at 128 reading none costs 1 % (499 -> 504 us for an 8192-token prompt).
    constexpr int PRE = D == 64 ? 0 : 2;
    uint4_t ka[PFK][2];
    const int i16 = lane & 15, bl = (lane & 31) >> 4;
    const int k_at = (ln % C::NG) * C::KG + (ln / C::NG) * C::ROWB + h2 * 16;
    const int v_at = (C::NG == 4 ? (i16 >> 2) * C::VG + h2 * C::ROWB : (4 * h2 + (i16 >> 2)) * C::VG) + (16 * bl + 4 * (i16 & 3)) * 2;
    constexpr int V_SLICE = 16 / C::NG * C::ROWB, V_PLUS8 = C::NG == 16 ? 8 * C::VG : 8 / C::NG * C::ROWB;
    auto read_k = [&](int kbase, int kb) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 2; t++) ka[kb % PFK][t] = *LDS_PTR(uint4_t, kbase + t * (32 / C::NG) * C::ROWB + kb * 32);
    };
    auto prefetch_k = [&](int i) __attribute__((always_inline)) {
        const int kbase = k_stage(tile_of(i)) + k_at;
#pragma unroll
        for (int kb = 0; kb < PRE; kb++) read_k(kbase, kb);
    };
    bool masked = false;  // the tile whose S^T was formed last is not wholly visible to this wavefront
    auto qk_pv = [&](int i, int at, auto do_qk, auto do_pv, auto prefetched) __attribute__((always_inline)) {
        constexpr bool QK = decltype(do_qk)::value, PV = decltype(do_pv)::value, PREFETCHED = decltype(prefetched)::value;
        const int kbase = k_stage(tile_of(i)) + k_at, vbase = v_stage(tile_of(i - 1)) + v_at;
        uint4_t va[2][NDB];
        auto read_v = [&](int gq) __attribute__((always_inline)) {  // gq = 2 t + kk: rows 16 gq + 4 h2 + {0..3} and + 8
#pragma unroll
            for (int db = 0; db < NDB; db++) {
                const int addr = vbase + gq * V_SLICE + db * 64;
                short4_t a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(short4_t, addr));
                short4_t a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(short4_t, addr + V_PLUS8));
                const uint2_t u0 = __builtin_bit_cast(uint2_t, a0), u1 = __builtin_bit_cast(uint2_t, a1);
                va[gq & 1][db] = uint4_t{u0[0], u0[1], u1[0], u1[1]};
            }
        };
        if constexpr (QK) {
#pragma unroll
            for (int kb = PREFETCHED ? PRE : 0; kb < PFK; kb++) read_k(kbase, kb);
#pragma unroll
            for (int kb = 0; kb < NKB; kb++) {
#pragma unroll
                for (int t = 0; t < 2; t++)
                    s[t] = Mma<T>::mfma(__builtin_bit_cast(vec8, ka[kb % PFK][t]), qreg[kb], kb == 0 ? zero16 : s[t]);
                if (kb + PFK < NKB) read_k(kbase, kb + PFK);
                if (PV && kb >= NKB - 4 && kb < NKB - 2) read_v(kb + 4 - NKB);
                load(at, kb);
                __builtin_amdgcn_sched_barrier(0);
            }
            const int j0 = j_begin + tile_of(i) * PF_BN;
            masked = !(j0 >= full_lo_w && j0 + PF_BN <= full_hi_w);
        } else {
            read_v(0);
            read_v(1);
        }
        if constexpr (PV) {
#pragma unroll
            for (int gq = 0; gq < 4; gq++) {
                const int t = gq >> 1, kk = gq & 1;
                const uint4_t braw = {pk[t][4 * kk], pk[t][4 * kk + 1], pk[t][4 * kk + 2], pk[t][4 * kk + 3]};
#pragma unroll
                for (int db = 0; db < NDB; db++)
                    o[db] = Mma<T>::mfma(__builtin_bit_cast(vec8, va[gq & 1][db]), __builtin_bit_cast(vec8, braw), o[db]);
                if (gq < 2) read_v(gq + 2);
                load(at, (QK ? NKB : 0) + gq);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int n = (QK ? NKB : 0) + (PV ? 4 : 0); n < PHASE_LOADS; n++) load(at, n);
    };
    // mask + online softmax (log2 domain, lazily rescaled) of tile i: s -> pk
    auto softmax = [&](int i) __attribute__((always_inline)) {
        if (masked) {
            const int j0 = j_begin + tile_of(i) * PF_BN;
            // element r of block t is key j0 + 32 t + 8 (r / 4) + 4 h2 + r % 4
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int key = j0 + 32 * t + 8 * (r >> 2) + 4 * h2 + (r & 3);
                    s[t][r] = (key >= klo && key < khi) ? s[t][r] : -INFINITY;
                }
        }
        // Probabilities against the reference the row already has; no maximum is taken.  The reference is whatever maximum
        // the row had when it was last set, so a probability may exceed 1: harmless while it stays inside the 16-bit
        // type's range (P is rounded to it for the second product; l and O are f32), and that is what the check below
        // guarantees: a lane's 32 probabilities are positive, so while their sum is at most 2^15 each of them is.
        auto probabilities = [&](float nm) __attribute__((always_inline)) {
            // four products ahead of the exponentials and two exponentials ahead of their uses: a lone wavefront has nothing
            // else to issue while one waits for the other
            constexpr int AHEAD = 4, LAG = 2;
            float x[32], sum[2] = {0.0f, 0.0f};
            auto scaled = [&](int r) __attribute__((always_inline)) { x[r] = __builtin_fmaf(s[r >> 4][r & 15], rr, nm); };
#pragma unroll
            for (int r = 0; r < AHEAD; r++) scaled(r);
#pragma unroll
            for (int r = 0; r < 32 + LAG; r++) {
                if (r < 32) x[r] = __builtin_amdgcn_exp2f(x[r]);
                if (r + AHEAD < 32) scaled(r + AHEAD);
                const int d = r - LAG;
                if (d >= 0) sum[d & 1] = d < 2 ? x[d] : sum[d & 1] + x[d];  // (a dot-product instruction would queue behind the MFMAs)
                if (d >= 0 && (d & 1)) pk[d >> 4][(d & 15) >> 1] = Mma<T>::pack2(x[d - 1], x[d]);
                __builtin_amdgcn_sched_barrier(0);
            }
            return sum[0] + sum[1];
        };
        float ts = probabilities(nmr);
        // Not at most 2^15 (which also catches the +inf and NaN a row without a reference produces): some row of the
        // wavefront needs its reference moved.  Take the tile's maximum, move every row's reference to at least that,
        // rescale what the row has accumulated, and form the tile's probabilities again.
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(ts <= 32768.0f)) != 0, 0)) {
            float mx = s[0][0];
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) mx = fmaxf(mx, s[t][r]);
            mx = half_swap_max(mx);
            const float m_new = fmaxf(m, mx);
            const float corr = (m == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f((m - m_new) * rr);
            m = m_new;
            l *= corr;
#pragma unroll
            for (int db = 0; db < D / 32; db++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[db][r] *= corr;
            // still no visible key: the tile's probabilities are exp2(-inf) = 0 and the row stays without a reference
            nmr = (m == -INFINITY) ? INFINITY : -m * rr;
            ts = probabilities((m == -INFINITY) ? 0.0f : nmr);
        }
        l += ts;
    };

    // ---- slot schedule ---------------------------------------------------------------------------------
    // Slots are separated by workgroup barriers.  Group 0 is in its matrix phase in even slots and in
    // its vector phase in odd slots; group 1 the other way round, one slot later.  Matrix phase of
    // tile i: S^T of tile i (reads K(i)), then P.V of tile i-1 (reads V(i-1)); K(i) is read in slots 2i - 1 (ahead, by
    // group 0) to 2i+1, V(i) in slots 2i+2 and 2i+3.  Vector phase: read the first K operands of the next matrix phase,
    // softmax, wait for a tile issued two matrix phases ago.
    // Tile t lives in stage t % 4.  In odd slot 2j+1 group 1 issues K(j+3) (its stage was last read for
    // K(j-1) in slot 2j-1) and makes sure in slot 2j+2 that K(j+2) has landed; in even slot 2j group 0 issues V(j+2)
    // (stage last read for V(j-2) in slot 2j-1) and makes sure in slot 2j+1 that V(j) has landed.  Every tile is thus
    // complete, and published by a barrier, before the slot of its first reader, and has had at least three
    // slots to arrive.
    // The tiles visible to a wavefront form one contiguous range [ia, ib).  Each group walks the slot
    // sequence in five static segments (nothing / first tile / steady state / last tile / nothing) so
    // that the steady-state loop body is branch-free and no state changes registers between phases.
    //
    // Key-split form (KS): both groups own the same 128 rows and group g takes the tiles t with t % 2 == g,
    // so a slot is the matrix phase of tile s for one group and the vector phase of tile s-1 for the other;
    // the groups' (m, l, O) are merged at the end.  K(t) is read in slot t (its first operands in
    // slot t-1), V(t) in slot t+2.  The group in its matrix phase in slot s issues K(s+4) into the stage K(s-1)
    // has just left (ring of 5) and V(s+1) into the stage of V(s-3), last read in slot s-1 (ring of 4), and
    // makes sure its loads of slot s-2, K(s+2) and V(s-1), have landed: each is published by a barrier
    // before the slot of its first reader and has had two slots to arrive.  The segments below then run on the
    // group's own tile count: local tile i of group g is tile 2 i + g.
    int ia = 0, ib = 0;
    if (wave_has_rows && hi_w > lo_w) {
        ia = (lo_w - j_begin) / PF_BN;
        ib = min(ntiles, (hi_w - j_begin + PF_BN - 1) / PF_BN);
        if (ib < ia) ib = ia;
    }
    int n_iter = ntiles + 1;  // iterations (two slots each) of either group
    if constexpr (KS) {
        ia = (ia + 1 - group) >> 1;  // this group's tiles below ia / below ib
        ib = (ib + 1 - group) >> 1;
        n_iter = (ntiles + 3) >> 1;
    }
    // MODE bit 0: S^T of tile i; bit 1: P.V of tile i-1; bit 2: softmax of tile i (group 0) / i-1 (group 1);
    // bit 3: the K operands of tile i were prefetched by the preceding vector phase;
    // bit 4: prefetch the K operands for the next matrix phase in the vector phase
    auto matrix_phase = [&](int i, int at, auto mode) __attribute__((always_inline)) {
        constexpr int MODE = decltype(mode)::value;
        __builtin_amdgcn_s_setprio(1);
        if constexpr ((MODE & 3) != 0)
            qk_pv(i, at, integral_constant<bool, (MODE & 1) != 0>{}, integral_constant<bool, (MODE & 2) != 0>{},
                  integral_constant<bool, (MODE & 8) != 0>{});
        else load_all(at);
        __builtin_amdgcn_s_setprio(0);
        if constexpr (KS) wait_loads(integral_constant<int, PHASE_LOADS>{});  // those of the matrix phase before have landed
    };
    // next_k: the tile whose S^T this wavefront computes in its next matrix phase
    auto vector_phase = [&](int i, int next_k, auto newer, auto mode) __attribute__((always_inline)) {
        constexpr int MODE = decltype(mode)::value;
        if constexpr ((MODE & 16) != 0) prefetch_k(next_k);
        if constexpr ((MODE & 4) != 0) softmax(i);
        if constexpr (!KS) wait_loads(newer);
    };
    // Between slots nothing but the barrier itself: no wavefront writes to LDS in the loop, and the K operands read ahead may
    // still be on their way (their stage is written two slots later at the earliest).
    auto slot_end = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto segment0 = [&](int i0, int i1, auto mode) __attribute__((always_inline)) {  // group 0: slot 2i matrix + V(i+2), slot 2i+1 vector
        for (int i = i0; i < i1; i++) {
            matrix_phase(i, KS ? 2 * i : i + 2, mode);
            slot_end();
            vector_phase(i, i + 1, integral_constant<int, 2 * C::LOADS>{}, mode);
            slot_end();
        }
    };
    auto segment1 = [&](int i0, int i1, auto mode) __attribute__((always_inline)) {  // group 1: slot 2i vector (tile i-1), slot 2i+1 matrix + K(i+3)
        for (int i = i0; i < i1; i++) {
            vector_phase(i - 1, i, integral_constant<int, C::LOADS>{}, mode);
            slot_end();
            matrix_phase(i, KS ? 2 * i + 1 : i + 3, mode);
            slot_end();
        }
    };
    if (ntiles > 0) {
        if constexpr (KS) {  // what slots -4 .. -1 would have issued
#pragma unroll
            for (int j = 0; j < C::LOADS; j++) {
                if (group == 0) issue_k(0, j), issue_k(2, j), issue_v(0, j);
                else issue_k(1, j), issue_k(3, j);
            }
        } else {
            // (tiles that are there: three of 64 keys at head_dim 128 cost a prompt of 18 rows 0.4 us of 8.5)
            load_all(0);
            if (ntiles > 1) load_all(1);
            if (moves_k && ntiles > 2) load_all(2);
        }
        if constexpr (FOLD) {
#pragma unroll
            for (int kb = 0; kb < QD / 16; kb++) qreg[kb] = Mma<T>::scaled(qreg[kb], pw);
        }
        wait_loads(integral_constant<int, 0>{});
        lds_barrier();
        if (group == 0) {
            // iteration i: S^T(i), softmax(i), P.V(i-1)
            segment0(0, ia, integral_constant<int, 0>{});
            if (ia < ib) {
                segment0(ia, ia + 1, integral_constant<int, 1 | 4 | 16>{});
                segment0(ia + 1, ib, integral_constant<int, 1 | 2 | 4 | 8 | 16>{});
                segment0(ib, ib + 1, integral_constant<int, 2>{});
                segment0(ib + 1, n_iter, integral_constant<int, 0>{});
            } else {
                segment0(ia, n_iter, integral_constant<int, 0>{});
            }
        } else {
            // iteration i: softmax(i-1), then S^T(i) and P.V(i-1)
            segment1(0, ia, integral_constant<int, 0>{});
            if (ia < ib) {
                segment1(ia, ia + 1, integral_constant<int, 1 | 8 | 16>{});
                segment1(ia + 1, ib, integral_constant<int, 1 | 2 | 4 | 8 | 16>{});
                segment1(ib, ib + 1, integral_constant<int, 2 | 4>{});
                segment1(ib + 1, n_iter, integral_constant<int, 0>{});
            } else {
                segment1(ia, n_iter, integral_constant<int, 0>{});
            }
        }
    }

    // the epilogue reuses the tile buffers: no tile load may still be on its way into them
    wait_loads(integral_constant<int, 0>{});
    lds_barrier();
    constexpr int SLICE = 32 * (D * 2 + 16);  // bytes per wavefront of the output transposition below
    if constexpr (KS) {
        // Group 1 hands its state to group 0, which holds the other half of the keys of the same rows:
        // log-sum-exp merge, as the split-KV combine does.  One f32 per lane per slot, above the slices the
        // output transposition uses.
        constexpr int PARK = 4 * SLICE;
        constexpr int NSLOT = D / 2 + 2;
        static_assert(PARK + NSLOT * 1024 <= C::LDS_BYTES, "merge area exceeds the tile buffers");
        auto park = (__attribute__((address_space(3))) float *)(lds_base + PARK) + (wave & 3) * 64 + lane;
        if (group == 1) {
#pragma unroll
            for (int db = 0; db < D / 32; db++)
#pragma unroll
                for (int r = 0; r < 16; r++) park[(db * 16 + r) * 256] = o[db][r];
            park[(D / 2) * 256] = m;
            park[(D / 2 + 1) * 256] = l;
        }
        lds_barrier();
        if (group == 1) return;
        const float m1 = park[(D / 2) * 256], l1 = park[(D / 2 + 1) * 256];
        const float mn = fmaxf(m, m1);
        const float c0 = (m == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f((m - mn) * rr);
        const float c1 = (m1 == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f((m1 - mn) * rr);
#pragma unroll
        for (int db = 0; db < D / 32; db++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[db][r] = o[db][r] * c0 + park[(db * 16 + r) * 256] * c1;
        l = l * c0 + l1 * c1;
        m = mn;
    }
    // ---- epilogue: out[query][dim] = O^T[dim][query] / l ----------------------------------------------
    const float l_tot = half_swap_sum(l);
    // With the keys split over workgroups the "output" is this share's row in the partials: O unnormalised
    // as f32 in 16-byte pieces, then (m, l); the merge kernel normalises.
    const bool parked = nks > 1;
    const float inv = parked ? 1.0f : 1.0f / l_tot;
    const bool dead = !parked && (l_tot == 0.0f);  // no visible key: the reference gives NaN (0/0)
    const bool out_f32 = parked || p.out_f32;
    const int64_t os0 = parked ? (int64_t)p.H * p.Sq * nks * p.pf_pitch : p.os[0];
    const int64_t os1 = parked ? (int64_t)p.Sq * nks * p.pf_pitch : p.os[1];
    const int64_t os2 = parked ? (int64_t)nks * p.pf_pitch : p.os[2];
    char *const og = parked ? (char *)(p.partials + (int64_t)ksplit * p.pf_pitch) : (char *)p.out;
    if (parked && query < p.Sq && h2 == 0) {
        float *ws = (float *)og + b * os0 + h * os1 + (int64_t)query * os2;
        ws[hd] = m * rr;  // base-2 exponent units
        ws[hd + 1] = l_tot;
    }
    if (out_vec || parked) {
        // transpose through a wavefront-private slice of the LDS so that every global store is a
        // 16-byte piece of a contiguous row; 32 rows per round for 2-byte outputs, 16 for f32
        const int esz = out_f32 ? 4 : 2;
        const int pitch = D * esz + 16;                      // rows stay 16-byte aligned, 4 banks apart
        static_assert(PF_WAVES * SLICE <= C::LDS_BYTES, "epilogue staging exceeds the tile buffers");
        auto wbase = lds_base + wave * SLICE;
        const int rounds = out_f32 ? 2 : 1;
        const int rows_per_round = 32 / rounds;
        const int cpr = D * esz / 16;
        for (int rd = 0; rd < rounds; rd++) {
            const int row_lo_ = rd * rows_per_round;
            if (ln >= row_lo_ && ln < row_lo_ + rows_per_round) {
#pragma unroll
                for (int db = 0; db < D / 32; db++)
#pragma unroll
                    for (int rq = 0; rq < 4; rq++) {
                        float v4[4];
#pragma unroll
                        for (int e = 0; e < 4; e++) v4[e] = dead ? __builtin_nanf("") : o[db][4 * rq + e] * inv;
                        const int dim = 32 * db + 8 * rq + 4 * h2;
                        if (out_f32) {
                            *(__attribute__((address_space(3))) float4_t *)(wbase + (ln - row_lo_) * pitch + dim * 4) =
                                float4_t{v4[0], v4[1], v4[2], v4[3]};
                        } else {
                            const uint2_t pk2 = {Mma<T>::pack2(v4[0], v4[1]), Mma<T>::pack2(v4[2], v4[3])};
                            *(__attribute__((address_space(3))) uint2_t *)(wbase + ln * pitch + dim * 2) = pk2;
                        }
                    }
            }
            wave_lds_sync();
            for (int c = lane; c < rows_per_round * cpr; c += 64) {
                const int row = c / cpr, col = c % cpr;
                const int qr = qw0 + row_lo_ + row;
                if (qr < p.Sq && (!PAD || col * 16 < hd * esz)) {
                    const uint4_t val = *(__attribute__((address_space(3))) uint4_t *)(wbase + row * pitch + col * 16);
                    const int64_t eidx = b * os0 + h * os1 + (int64_t)qr * os2;
                    *(uint4_t *)(og + eidx * esz + col * 16) = val;
                }
            }
            wave_lds_sync();
        }
    } else if (query < p.Sq) {
        const int64_t obase = b * p.os[0] + h * p.os[1] + (int64_t)query * p.os[2];
#pragma unroll
        for (int db = 0; db < D / 32; db++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int dim = 32 * db + 8 * (r >> 2) + 4 * h2 + (r & 3);
                if (PAD && dim >= hd) continue;
                const float val = dead ? __builtin_nanf("") : o[db][r] * inv;
                if (p.out_f32) ((float *)p.out)[obase + dim * p.os[3]] = val;
                else ((T *)p.out)[obase + dim * p.os[3]] = from_float<T>(val);
            }
    }
}

// Query blocks of 256 rows leave CUs idle when there are few of them (short prompts, a few new rows on a long
// cache), and a causal prompt's last blocks are several times longer than its first.  The key-split form (128
// rows, twice the workgroups, the longest one half as long) costs about 11 % per tile (f16, 32/8 heads at 128, 8192-token
// prompt: 535 us against 481) and a longer prologue and epilogue; measured, it wins while the 256-row grid fills at most half the CUs (8 to 32
// heads, 1024 to 2049 rows: 1.25 - 1.5 x), for up to 128 query rows (where the second wavefront group would have no
// rows at all; 1.07 x at 128, 1.15 at 64), and, where later rows see more keys than earlier ones, for one workgroup per CU
// when a head has 8 or more query blocks; it loses with fewer than three key tiles.
// For one workgroup per CU the 256-row form takes as long as its longest block, the key-split form about a quarter more than the
// mean one (two of its workgroups follow each other on a CU).  f16, us a call, 256-row and key-split form on one card: without a
// mask, 16 heads, head_dim 80, 4096 x 4096 keys 90 and 99, 3000 57 and 66; 64, 2500 40 and 49; 128, 2500 58 and 76, 4096 122 and 136;
// causal, 128, 32/8 heads, 2048 rows on 2048 keys 50 and 47, 4096 106.1 and 105.5, 5120 133.8 and 136.2, 8192 218 and 227; 24/8
// heads 46 and 39, on 4096 keys 91 and 88, 5120 113.2 and 112.9, 6144 136 and 138; 16/8 heads, 3000 rows on 3000 keys 61 and 48, 6000 125
// and 121, 7500 158.2 and 157.4, 9000 190 and 193.  So rows that all see the same keys keep the 256-row form, and where they see
// the keys up to their own position the line is 2.5 keys per row.  Under a window narrower than that it stays at 2, beyond which
// the 256-row form wins by more (2048 rows on 4096 keys under a window of 2048: 68 and 78).  Rows with half a window or more behind the
// first of them see about the same keys as well, however few the call as a whole sees (12/12 heads at 128, 3132 rows under 2512 68 and 85,
// at 80, two sequences of 1939 under 208 22 and 26), but where the key-split form has one workgroup per CU, or little more and the first rows see less
// than a window (12/12 at 128, 2668 behind 226 under 452 29 and 20; 8/4 at 64, 4130 behind 1313 under 2626 50 and 41).  Sequences of different lengths in
// a batch are even grids in this sense (2 to 8 of them, 500 to 2048 keys long: 0.80 to 0.85 of the key-split form's time).
// later_rows_see: the keys up to the last row's own where rows see the keys up to their own position, 0 where all see the same.
int prefill_mfma_block_rows(int B, int H, int Sq, int Skv, int key_shares, int64_t later_rows_see, int64_t window, int compute_units) {
    const int nqb = (Sq + PF_BM - 1) / PF_BM;
    const long wgs = (long)nqb * B * H * (key_shares > 1 ? key_shares : 1);
    if (Skv <= 2 * PF_BN) return PF_BM;
    if (Sq <= PF_BM / 2 || 2 * wgs <= compute_units) return PF_BM / 2;
    if (wgs > compute_units || nqb < 8 || later_rows_see <= 0) return PF_BM;
    const int64_t keys = later_rows_see < Skv ? later_rows_see : Skv;
    const bool narrow = window > 0 && window < keys;
    const long of_half = (long)((Sq + PF_BM / 2 - 1) / (PF_BM / 2)) * B * H;
    const int64_t before = later_rows_see - Sq + 1;  // keys that the first row sees without the window
    // (before < window + 128: the keys begin where the first row's window does; they do not where the call brings lengths)
    if (narrow && window <= Sq && before < window + 128 &&
        (before >= window ? of_half > compute_units : 2 * before >= window && 4 * of_half > 5L * compute_units))
        return PF_BM;
    return 2L * Sq > Skv || (!narrow && 5L * Sq >= 2 * keys) ? PF_BM / 2 : PF_BM;
}

// Head dims 64, 96 and 128 are this kernel's own.  The other multiples of 8 above 64 run on it padded, quicker than on the
// wide-head kernel, whose wavefronts read every LDS operand for half as many matrix instructions (both in turn on one card, us a
// call; f16, 16 heads, 4096 x 4096 keys without a mask: head_dim 72 147 -> 120, 80 150 -> 124, 88 163 -> 130, 104 196 -> 136, 112
// 202 -> 144, 120 201 -> 147; causal, 80: 157 -> 75 (two of that kernel's 128-row blocks per CU wait for the longest); 512-token
// causal prompt, 32/8 heads, 80: 17.0 -> 15.9).  Below 64 the padding costs what the kernel gains unless the grid fills the
// chip (head_dim 40: 4096 keys 134 -> 104; head_dim 32: 116 -> 102), and to 32, where it is half of the work or more, also in
// short row blocks (300 rows of four sequences 60 -> 64).
bool prefill_mfma_rows256_takes(int D, float scale, int B, int H, int Sq, int compute_units) {
    if (!(D % 8 == 0 && D >= 8 && D <= 128 && scale > 0.0f && scale * PF_LOG2E < 2.0f)) return false;
    if (D >= 64) return true;
    const long blocks = (long)B * H * ((Sq + PF_BM - 1) / PF_BM);
    return blocks >= compute_units && (D > 32 || Sq >= 1024);
}

template <typename T>
static int launch_t(const AttnParams &p0, hipStream_t stream) {
    AttnParams p = p0;
    const int cus = p.cus > 0 ? p.cus : 256;
    const int64_t later_rows_see = p.analytic && p.causal ? p.q_pos_offset + p.Sq : p.mask_kind == FHIP_MASK_QK ? p.Skv : 0;
    const int bm = prefill_mfma_block_rows(p.B, p.H, p.Sq, p.Skv, p.pf_nsplit, later_rows_see, p.analytic ? p.window : 0, cus);
    const bool ks = bm == PF_BM / 2;
    p.pf_pack = ks ? prefill_mfma_pack(p.B, p.H, p.G, p.Sq, p.Skv, cus) : 0;
    const int nqb = p.pf_pack ? 1 : (p.Sq + bm - 1) / bm;
    const long blocks = (long)nqb * p.B * (p.pf_pack ? p.H / 4 : p.H) * (p.pf_nsplit > 1 ? p.pf_nsplit : 1);
    if (blocks > 0x7fffffffL) {
        set_error("prefill: too many workgroups (%ld)", blocks);
        return FHIP_ERR_UNSUPPORTED;
    }
    dim3 grid((unsigned)blocks), block(64 * PF_WAVES);
    // rows of the output can be written in 16-byte pieces when they are contiguous and aligned
    const int oeb = p.out_f32 ? 4 : 2;
    int out_vec = (p.os[3] == 1 || p.D == 1) && ((uintptr_t)p.out % 16 == 0);
    for (int i = 0; i < 3; i++)
        if ((p.os[i] * oeb) % 16 != 0) out_vec = 0;
#define PF_LAUNCH(DIM, QDIM, PAD)                                                                               \
    if (ks) FHIP_LAUNCH_MAIN((prefill_mfma_kernel<T, DIM, QDIM, PAD, true>), grid, block, stream, p, p, nqb, out_vec); \
    else FHIP_LAUNCH_MAIN((prefill_mfma_kernel<T, DIM, QDIM, PAD, false>), grid, block, stream, p, p, nqb, out_vec)
    if (p.D % 8 != 0 || p.D < 8 || p.D > 128) {
        set_error("prefill MFMA kernel: head_dim %d is not a multiple of 8 up to 128", p.D);
        return FHIP_ERR_UNSUPPORTED;
    }
    if (p.D == 64) { PF_LAUNCH(64, 64, false); }
    else if (p.D == 96) { PF_LAUNCH(96, 96, false); }
    else if (p.D == 128) { PF_LAUNCH(128, 128, false); }
    else if (p.D < 64) { PF_LAUNCH(64, 64, true); }
    else if (p.D <= 80) { PF_LAUNCH(96, 80, true); }
    else if (p.D < 96) { PF_LAUNCH(96, 96, true); }
    else if (p.D <= 112) { PF_LAUNCH(128, 112, true); }
    else { PF_LAUNCH(128, 128, true); }
#undef PF_LAUNCH
    FHIP_HIP_CHECK(hipGetLastError());
    if (p.pf_nsplit > 1) return launch_prefill_merge(p, sizeof(T) == 2 && std::is_same<T, half_t>::value ? FHIP_F16 : FHIP_BF16, stream);
    return FHIP_OK;
}

// Few query rows on a long cache: 256-row query blocks alone leave most CUs idle, so the keys are split over
// workgroups too, down to 1024 keys per share, until there are about two workgroups per CU.
// Query heads per workgroup of the packed form (0: not packed).  Packing divides the workgroups by four, and a share of
// the keys is at least 1024 keys long, so it is taken when the packed grid still reaches half the CUs (12..32 rows:
// batch 8 on 8192 keys 98 -> 66..81 us, batch 4 on 4096 keys 45 -> 28 us, batch 1 on 32768 keys 68 -> 40 us; with a
// quarter of the CUs, batch 1 on 8192 keys, the unpacked grid is as quick: 25.7 against 26.5 us).
int prefill_mfma_pack(int B, int H, int G, int Sq, int Skv, int compute_units) {
    if (!(Sq <= 32 && G >= 4 && G % 4 == 0) || Skv <= 2 * PF_BN) return 0;
    const long shares = Skv / 1024 > 1 ? Skv / 1024 : 1;
    return 2 * (long)B * (H / 4) * shares >= compute_units ? 4 : 0;
}

// Time of a call in us, by the form it takes in that many shares: rounds of workgroups that walk their tiles, and parking and
// merging the shares.  Constants fitted to 140 random calls (chunks, turns and images of 8 to 32 heads at 64 to 128 dims, each in both
// forms and up to 48 shares): 10 % off in the mean square.
static double prefill_mfma_time(int B, int H, int G, int Sq, int Skv, int D, int64_t later_rows_see, int64_t window, int compute_units, int ns) {
    const int c = ((Skv + ns - 1) / ns + PF_BN - 1) / PF_BN * PF_BN, n = (Skv + c - 1) / c;
    const int bm = prefill_mfma_block_rows(B, H, Sq, Skv, n, later_rows_see, window, compute_units);
    const bool ks = bm == PF_BM / 2, packed = ks && prefill_mfma_pack(B, H, G, Sq, Skv, compute_units);
    const long wgs = (long)B * (packed ? H / 4 : H) * ((Sq + bm - 1) / bm) * n, rounds = (wgs + compute_units - 1) / compute_units;
    const double dims = D <= 64 ? 1.0 : D <= 96 ? 1.43 : 1.86;
    double us = 4.6 + rounds * (ks ? 5.3 + 0.356 * dims * (c / PF_BN) : 3.9 + 0.579 * dims * (c / PF_BN));
    if (n > 1) us += 3.0 + 0.488e-6 * prefill_mfma_workspace_bytes(B, H, Sq, D, n);
    return us;
}

// uneven: a square call whose rows see the keys up to their own position (a mask tensor is taken for one): by the rules alone.
// later_rows_see, window: as for prefill_mfma_block_rows.
void prefill_mfma_plan(int B, int H, int G, int Sq, int Skv, int D, bool causal_square, bool uneven, int64_t later_rows_see, int64_t window,
                       bool unknown_lengths, int compute_units, int *nsplit, int *chunk) {
    *nsplit = 1;
    *chunk = Skv;
    if (causal_square) return;
    const long wgs = (long)B * (prefill_mfma_pack(B, H, G, Sq, Skv, compute_units) ? H / 4 : H) * ((Sq + PF_BM - 1) / PF_BM);
    if (wgs == 0) return;
    // By rule a grid of query blocks that keeps half the chip busy by itself is not split (the times below may find otherwise).
    const long want = (2L * compute_units + wgs - 1) / wgs;
    long most = Skv / 1024;
    // A few rows on a short cache: shares down to 512 keys, and for up to 64 rows to 256, while CUs would stay without a
    // workgroup (f16, 32/8 heads, head_dim 128, B1: 12...32 rows on 2048 keys 24.6 -> 17.8 us, on 4096 keys 24.7 -> 20.7;
    // 128 rows on 2048 keys 28.8 -> 25.7).  On 1024 keys two shares of 512 lose with more than 64 rows (21.2 -> 23.4 us).
    const bool few_rows = 2L * Sq <= Skv && (Sq <= 64 || Skv >= 2048);
    if (few_rows && (want < most ? want : most) * wgs < compute_units) most = Skv / 512;
    if (few_rows && Sq <= 64 && (want < most ? want : most) * wgs < compute_units) most = Skv / 256;
    long ns = 2 * wgs > compute_units ? 1 : want < most ? want : most;
    if (ns < 1) ns = 1;
    // These rules count workgroups and not their rounds, nor the bytes of the partials: the shares of least time by the function
    // above, the fewest within 1 % of it, are taken where that is 5 % less than the rules' (shares_gain), or 10 % for grids that the rules do not split
    // (us a call: four sequences of 207 rows of 32/8 heads at 96 under a window of 4096 84 -> 56 in none; 189 rows of 8/4 heads at 80 on 1993 keys 23.5 -> 19, 231 of 32/8 at 64 on 14900
    // 59 -> 48, 49 of 32/32 at 128 on 3032 36 -> 22; over 500 random calls without lengths or a mask tensor 0.93 of the rules' time, the
    // worst 1.11; at 5 % everywhere large ones lost up to 14 %: 32/32 heads at 80, 2859 rows on 7370 keys 209 and 238).
    constexpr int SHARES[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 28, 32, 40, 48};
    double times[sizeof(SHARES) / sizeof(SHARES[0])], least = 0.0;
    int tried = 0;
    for (const int n : SHARES) {
        if (uneven) break;
        // (three rounds gain nothing more; partials of at most 64 MiB)
        if (n > 1 && (Skv / n < 128 || (n - 1) * wgs > 3L * compute_units || prefill_mfma_workspace_bytes(B, H, Sq, D, n) > ((size_t)64 << 20)))
            break;
        times[tried] = prefill_mfma_time(B, H, G, Sq, Skv, D, later_rows_see, window, compute_units, n);
        if (tried == 0 || times[tried] < least) least = times[tried];
        tried++;
    }
    for (int i = 0; i < tried; i++) {
        if (times[i] > 1.01 * least) continue;
        const double gain = std::min(shares_gain(unknown_lengths), 2 * wgs > compute_units ? 0.9 : 1.0);
        if (times[i] < gain * prefill_mfma_time(B, H, G, Sq, Skv, D, later_rows_see, window, compute_units, (int)ns)) ns = SHARES[i];
        break;
    }
    if (ns < 2) return;
    long c = (Skv + ns - 1) / ns;
    c = (c + PF_BN - 1) / PF_BN * PF_BN;
    *chunk = (int)c;
    *nsplit = (int)((Skv + c - 1) / c);
}

size_t prefill_mfma_workspace_bytes(int B, int H, int Sq, int D, int nsplit) {
    if (nsplit <= 1) return 0;
    return (size_t)B * H * Sq * nsplit * (size_t)(D + 4) * sizeof(float);
}

int launch_prefill_mfma(const AttnParams &p, fhip_dtype dtype, hipStream_t stream) {
    if (dtype == FHIP_F16) return launch_t<half_t>(p, stream);
    if (dtype == FHIP_BF16) return launch_t<bf16_t>(p, stream);
    set_error("prefill MFMA kernel takes f16/bf16 only");
    return FHIP_ERR_UNSUPPORTED;
}

}  // namespace fhip
