// Prefill attention in f32 precision on the gfx950 f32 matrix instruction (v_mfma_f32_32x32x2_f32): calls that
// attn_prefill_f32_terms.hip cannot address (prefill_f32_terms_takes): K or V rows that overlap, a K, V
// or Q slice of 2 GiB and more, or grids beyond its dimensions; and above head_dim 128
// 16-bit tensors, short calls of few rows and unsplit ones whose rows see few keys (wide_in_terms, wide_f32_time).
//
// A workgroup of 4 wavefronts owns 128 query rows of one (batch, head), a wavefront 32 of them; K/V tiles of 32 rows pass
// through LDS.
//   S^T (32 keys x 32 queries) = K_tile . Q^T   A = K[key][dim] from LDS (128-bit reads, the four
//                                               values feed four MFMA steps), B = Q in registers
//   softmax down the key axis: every lane owns one query and 16 keys -> in-lane folds plus one
//   exchange with the lane 32 away
//   O^T (D x 32 queries) += V^T . P^T           A = V[key][dim] read row-major (one f32 per lane),
//                                               B = the S^T accumulator registers themselves
// Products and sums are f32 throughout.  Also here: the plan of a call's key split for all f32 kernels, and the kernel that
// merges the shares.
//
// Reference semantics: fusor-ml/fusor/src/composite/flash_attention.rs:141-199; this is the data
// type kalosm-llama always calls with (models/kalosm-llama/src/raw/attention_layer.rs:400-448).
#include <algorithm>
#include <type_traits>

#include "attn_bounds.h"
#include "attn_f32.h"
#include "common.h"
#include "device_utils.h"

namespace fhip {

constexpr int PF32_WAVES = 4;
constexpr int PF32_BN = 32;
#define LDS32_PTR(type, byte_off) ((__attribute__((address_space(3))) type *)(lds_base + (byte_off)))

template <typename T, int D, int MODE>
__global__ __launch_bounds__(64 * PF32_WAVES, 2) void prefill_f32_kernel(AttnParams p, int nqb) {
    constexpr bool BIAS = MODE != PF32_INTERVALS;  // the mask-adding code is in the kernel
    constexpr int BM = 32 * PF32_WAVES;   // query rows per workgroup
    // Which head dims a 32-row block of O^T holds.  With 2 or 4 blocks, row i of block db is dim NDB i + db: the
    // V operands of all blocks for one key then sit side by side and one 8- or 16-byte LDS read feeds NDB matrix
    // instructions (a 4-byte read per instruction leaves a lone wavefront waiting on LDS latency most of the time).
    constexpr int NDB = D / 32;
    constexpr bool PACKED = (NDB == 2 || NDB == 4);
    auto dim_of = [](int db, int i) __attribute__((always_inline)) { return PACKED ? NDB * i + db : 32 * db + i; };
    constexpr int KP = D * 4 + 16;  // row pitch in bytes: rows 4 banks apart -> conflict-free b128 reads
    constexpr int K_BYTES = PF32_BN * KP;
    constexpr int CPR = D / 4;      // 16-byte chunks per row
    constexpr int GT = 64 * PF32_WAVES;
    constexpr int NCH = PF32_BN * CPR / GT;
    static_assert(PF32_BN * CPR % GT == 0, "the threads must cover a tile evenly");
    __shared__ __attribute__((aligned(16))) char smem[2 * K_BYTES];
    auto lds_base = (__attribute__((address_space(3))) char *)smem;

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

    const int bh_count = p.B * p.H;
    const int nks = max(p.pf_nsplit, 1);
    const int ksplit = blockIdx.x % nks;  // which share of the keys (0 when the keys are not split over workgroups)
    const int id = blockIdx.x / nks;
    const int qb = nqb - 1 - id / bh_count;
    int rem = id % bh_count;
    const int b = rem / p.H;
    int h = rem % p.H;
    if ((p.H & 7) == 0) h = (h & 7) * (p.H >> 3) + (h >> 3);
    const int g = h / p.G;
    // Rows of a tile beyond the sequence's own keys (kv_lens below the view's length: a ragged batch in one cache
    // allocation) are never fetched: what such rows hold, NaN included, must not reach the result as 0 x NaN in P . V.
    // (likewise the rows behind the last query's own position when the call says where its rows stand inside a longer
    // cache view: a causal descriptor with q_pos_offset + Sq below the view's length)
    int key_end = p.kv_lens ? min(p.Skv, max(p.kv_lens[b], 1)) : p.Skv;
    if (p.analytic && p.causal) key_end = (int)min((int64_t)key_end, max(p.q_pos_offset + p.Sq, (int64_t)1));

    const int q0 = qb * BM;
    const int qw0 = q0 + 32 * wave;
    const int query = qw0 + ln;
    // Q operand: Q[query][8 kc + 4 h2 .. +4]; requested before the bounds, whose table reads (mask tensors) would
    // otherwise delay these loads by a memory latency
    float4_t qreg[D / 8];
    {
        const int qrow = min(query, p.Sq - 1);
        const T *qp = (const T *)p.q + b * p.qs[0] + h * p.qs[1] + (int64_t)qrow * p.qs[2];
#pragma unroll
        for (int kc = 0; kc < D / 8; kc++)
            qreg[kc] = 8 * kc + 4 * h2 < p.D ? load4(qp + 8 * kc + 4 * h2) : float4_t{0.f, 0.f, 0.f, 0.f};
    }
    // uniform over the launch
    const bool bias_on = MODE == PF32_BIAS || (MODE == PF32_EITHER && *p.iv_bad == p.bad_tag);
    RowBounds rb = row_bounds(p, MODE == PF32_BIAS ? nullptr : p.iv, b, q0, BM, qw0, lane);
    if constexpr (MODE == PF32_EITHER) {
        // the table was read whatever the scan found (its loads need not wait for that word); without the interval
        // form the bounds are those of a call whose mask is added
        if (bias_on) rb = row_bounds(p, nullptr, b, q0, BM, qw0, lane);
    }
    if (nks > 1) {  // this workgroup's share of the keys
        const int c_lo = ksplit * p.pf_chunk, c_hi = c_lo + p.pf_chunk;
        rb.lo_wg = max(rb.lo_wg, c_lo), rb.hi_wg = min(rb.hi_wg, c_hi);
        rb.lo_w = max(rb.lo_w, c_lo), rb.hi_w = min(rb.hi_w, c_hi);
        rb.full_lo_w = max(rb.full_lo_w, c_lo), rb.full_hi_w = min(rb.full_hi_w, c_hi);
        rb.klo = max(rb.klo, c_lo), rb.khi = min(rb.khi, c_hi);
    }
    const int lo_wg = rb.lo_wg, hi_wg = rb.hi_wg, lo_w = rb.lo_w, hi_w = rb.hi_w;
    const bool wave_has_rows = qw0 < p.Sq;

    const T *kg = (const T *)p.k + b * p.ks[0] + g * p.ks[1];
    const T *vg = (const T *)p.v + b * p.vs[0] + g * p.vs[1];

    float16_t o[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[db][r] = 0.0f;
    float m = -INFINITY, l = 0.0f;
    // scores reach the softmax in the base-2 domain: raw dot products times scale * log2(e); with BIAS they are
    // scaled, biased, and multiplied by log2(e) where probabilities are formed (see `probability` in attn_f32.h)
    const float scale2 = bias_on ? PF32_LOG2E : p.scale * PF32_LOG2E, log2_unit = bias_on ? PF32_LOG2E : 1.0f;
    const T *mrow = nullptr;
    if constexpr (BIAS)
        mrow = (const T *)p.mask + (int64_t)(p.mask_kind == FHIP_MASK_QK ? min(query, p.Sq - 1) : b) * p.ms0;

    const int j_begin = (lo_wg / PF32_BN) * PF32_BN;
    const int ntiles = hi_wg > j_begin ? (hi_wg - j_begin + PF32_BN - 1) / PF32_BN : 0;
    // a thread's chunks of a tile are a fixed number of rows apart when the threads cover whole rows
    constexpr bool AFFINE = (GT % CPR == 0);
    constexpr int RSTEP = AFFINE ? GT / CPR : 0;
    const bool whole_rows = p.D == D;

    // One tile's math: S^T from the K image, online softmax, then O^T += V^T . P^T from the V image
    auto tile_math = [&](int j0) __attribute__((always_inline)) {
        float bias[BIAS ? 16 : 1];
        if constexpr (BIAS) {  // requested before the matrix work that hides their latency
            if (bias_on) {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int key = j0 + 8 * (r >> 2) + 4 * h2 + (r & 3);
                    bias[r] = key < p.Skv ? to_float(mrow[(int64_t)key * p.ms1]) : 0.0f;
                }
            }
        }

        // S^T: contraction step (kc, i) uses dim 8 kc + 4 h2 + i on both operands
        float16_t s;
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = 0.0f;
#pragma unroll
        for (int kc = 0; kc < D / 8; kc++) {
            const float4_t a = *LDS32_PTR(float4_t, ln * KP + (8 * kc + 4 * h2) * 4);
#pragma unroll
            for (int i = 0; i < 4; i++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], qreg[kc][i], s, 0, 0, 0);
        }

        // element r is key j0 + 8 (r / 4) + 4 h2 + r % 4 for query `query`
        if (!(j0 >= rb.full_lo_w && j0 + PF32_BN <= rb.full_hi_w)) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int key = j0 + 8 * (r >> 2) + 4 * h2 + (r & 3);
                s[r] = (key >= rb.klo && key < rb.khi) ? s[r] : -INFINITY;
            }
        }

        if constexpr (BIAS) {
            if (bias_on) {
#pragma unroll
                for (int r = 0; r < 16; r++) s[r] = s[r] * p.scale + bias[r];
            }
        }

        float mx = s[0];
#pragma unroll
        for (int r = 1; r < 16; r++) mx = fmaxf(mx, s[r]);
        mx = half_swap_max32(mx);
        const float m_new = fmaxf(m, bias_on ? mx : mx * scale2);
        const float corr = moved_reference(m, m_new, log2_unit);
        m = m_new;
        const float m2 = m * log2_unit, m_safe = (m2 == -INFINITY) ? 0.0f : m2;
        // rows that have seen nothing but lowest values: those equal to the reference count
        const float lowest = bias_on && m2 == -INFINITY && m > -INFINITY ? m : __builtin_nanf("");
        float psum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const float pr = __builtin_amdgcn_exp2f(fmaf(s[r], scale2, -m_safe));
            s[r] = BIAS && s[r] == lowest ? 1.0f : pr;
            psum += s[r];
        }
        l = l * corr + psum;
#pragma unroll
        for (int db = 0; db < D / 32; db++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[db][r] *= corr;

        // O^T += V^T . P^T: contraction step r pairs this half-wave's key 8 (r/4) + 4 h2 + r%4
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int krow = 8 * (r >> 2) + 4 * h2 + (r & 3);
            if constexpr (NDB == 4) {
                const float4_t a = *LDS32_PTR(float4_t, K_BYTES + krow * KP + ln * 16);
#pragma unroll
                for (int db = 0; db < 4; db++) o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[db], s[r], o[db], 0, 0, 0);
            } else if constexpr (NDB == 2) {
                typedef float float2_t __attribute__((ext_vector_type(2)));
                const float2_t a = *LDS32_PTR(float2_t, K_BYTES + krow * KP + ln * 8);
#pragma unroll
                for (int db = 0; db < 2; db++) o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[db], s[r], o[db], 0, 0, 0);
            } else {
#pragma unroll
                for (int db = 0; db < NDB; db++) {
                    const float a = *LDS32_PTR(float, K_BYTES + krow * KP + (32 * db + ln) * 4);
                    o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, s[r], o[db], 0, 0, 0);
                }
            }
        }
    };

    float4_t kst[NCH], vst[NCH];
    auto load_tile = [&](int j0) {
        if (AFFINE && whole_rows && j0 + PF32_BN <= key_end) {
            // a tile inside the key axis with rows as wide as the kernel's: one address per thread, the chunks a fixed
            // number of rows apart
            const T *pk = kg + (int64_t)(j0 + tid / CPR) * p.ks[2] + (tid % CPR) * 4;
            const T *pv = vg + (int64_t)(j0 + tid / CPR) * p.vs[2] + (tid % CPR) * 4;
            const int64_t kstep = (int64_t)RSTEP * p.ks[2], vstep = (int64_t)RSTEP * p.vs[2];
#pragma unroll
            for (int i = 0; i < NCH; i++) {
                kst[i] = load4(pk + i * kstep);
                vst[i] = load4(pv + i * vstep);
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < NCH; i++) {
            const int cid = tid + GT * i;
            const int row = cid / CPR, col = cid % CPR;
            const int key = min(j0 + row, key_end - 1);
            const bool in_row = col * 4 < p.D;  // a head_dim below D is padded with zeros
            kst[i] = in_row ? load4(kg + (int64_t)key * p.ks[2] + col * 4) : float4_t{0.f, 0.f, 0.f, 0.f};
            vst[i] = in_row ? load4(vg + (int64_t)key * p.vs[2] + col * 4) : float4_t{0.f, 0.f, 0.f, 0.f};
        }
    };
    auto store_tile = [&]() {
#pragma unroll
        for (int i = 0; i < NCH; i++) {
            const int cid = tid + GT * i;
            const int row = cid / CPR, col = cid % CPR;
            *LDS32_PTR(float4_t, row * KP + col * 16) = kst[i];
            *LDS32_PTR(float4_t, K_BYTES + row * KP + col * 16) = vst[i];
        }
    };

    if (ntiles > 0) load_tile(j_begin);

    for (int t = 0; t < ntiles; t++) {
        const int j0 = j_begin + t * PF32_BN;
        lds_barrier();  // everyone finished reading the previous tile (LDS-only barrier: the prefetch
        store_tile();   // issued below stays in flight across the math)
        lds_barrier();
        if (t + 1 < ntiles) load_tile(j0 + PF32_BN);

        const bool tile_visible = wave_has_rows && j0 < hi_w && j0 + PF32_BN > lo_w;
        if (!tile_visible) continue;
        tile_math(j0);
    }

    const float l_tot = half_swap_sum32(l);
    if (nks > 1) {
        // park this share's state; the merge kernel normalises
        if (query < p.Sq) {
            float *ws = p.partials + ((((int64_t)b * p.H + h) * p.Sq + query) * nks + ksplit) * p.pf_pitch;
#pragma unroll
            for (int db = 0; db < D / 32; db++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int dim = dim_of(db, 8 * (r >> 2) + 4 * h2 + (r & 3));
                    if (dim < p.D) ws[dim] = o[db][r];
                }
            if (h2 == 0) {
                ws[p.D] = m;
                ws[p.D + 1] = bias_on ? -l_tot : l_tot;  // (the sign tells the merge kernel m's unit)
            }
        }
        return;
    }
    if (query < p.Sq) {
        const int64_t ob = b * p.os[0] + h * p.os[1] + (int64_t)query * p.os[2];
#pragma unroll
        for (int db = 0; db < D / 32; db++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int dim = dim_of(db, 8 * (r >> 2) + 4 * h2 + (r & 3));
                if (dim < p.D) store_out<T>(p, ob + dim * p.os[3], o[db][r] / l_tot);  // no visible key: 0/0 = NaN like the reference
            }
    }
}

// Merge of the key shares: a log-sum-exp over the shares of each (batch, head, query row), then the division the
// single-pass form does in its epilogue.  A row's references m are exponents of two, or, where a mask is added to the
// scores, in the scores' own units: those rows' sums l are parked with their sign set (-0.0 included).
// LPR lanes share a row, four dims each: a share is one load of four values and one of (m, l).
// Bound: the memory latency of a round of eight shares, and the partials' bytes where there are many.  With one wavefront per row and
// six loads per share 16-bit calls in two to eight shares took 1.04 to 1.09 times as long in all, f32 ones 1.03.
typedef float4_t __attribute__((aligned(8))) float4_at8_t;  // a row of the partials is D + 2 or D + 4 floats
typedef float float2_at8_t __attribute__((ext_vector_type(2)));
template <typename T, int LPR>
__global__ __launch_bounds__(256) void prefill_f32_merge_kernel(AttnParams p, int out_vec) {
    request_arguments<AttnParams>();
    const int64_t row = (int64_t)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
    const int D = p.D, dim = 4 * (threadIdx.x % LPR);
    const int64_t rows = (int64_t)p.B * p.H * p.Sq;
    if (row >= rows || dim >= D) return;
    // the same hand-over between the interval form and the mask-adding form as in the main kernel (none when the
    // main kernel held both forms)
    if (!p.iv_either && ((p.iv_bad && *p.iv_bad == p.bad_tag) || (p.only_if_bad && *p.only_if_bad != p.bad_tag))) return;
    const int ns = p.pf_nsplit, pitch = p.pf_pitch;
    const float *ws = p.partials + row * ns * pitch;
    // eight shares per round of loads (a round costs one memory latency)
    float M = -INFINITY, L = 0.0f;
    float4_t A = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s0 = 0; s0 < ns; s0 += 8) {
        float ms[8], ls[8];
        float4_t av[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const bool ok = s0 + u < ns;
            const float *src = ws + (ok ? s0 + u : s0) * pitch;
            const float2_at8_t ml = *(const float2_at8_t *)(src + D);
            av[u] = *(const float4_at8_t *)(src + dim);
            ms[u] = ok ? ml[0] : -INFINITY;
            ls[u] = ok ? ml[1] : 0.0f;
            if (!ok) av[u] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
        float Mn = M;
#pragma unroll
        for (int u = 0; u < 8; u++) Mn = fmaxf(Mn, ms[u]);
        // as moved_reference (attn_f32.h) does it; nothing here waits for a single load of the round
        const float unit = __float_as_int(ls[0]) < 0 ? PF32_LOG2E : 1.0f, M2 = Mn * unit, Ms = M2 == -INFINITY ? 0.0f : M2;
        float c, w[8];
        {
#pragma clang fp contract(off)
            c = __builtin_amdgcn_exp2f(M * unit - Ms);
#pragma unroll
            for (int u = 0; u < 8; u++) w[u] = __builtin_amdgcn_exp2f(ms[u] * unit - Ms);
        }
        if (M2 == -INFINITY && Mn > -INFINITY) {
            c = M == Mn ? 1.0f : 0.0f;
#pragma unroll
            for (int u = 0; u < 8; u++) w[u] = ms[u] == Mn ? 1.0f : 0.0f;
        }
        L *= c;
        A *= c;
#pragma unroll
        for (int u = 0; u < 8; u++) {
            L += w[u] * ls[u];
#pragma unroll
            for (int e = 0; e < 4; e++) A[e] += w[u] * av[u][e];
        }
        M = Mn;
    }
    L = fabsf(L);
    int64_t at;  // of the row in the result
    if (rows <= 0x7fffffff) {
        const uint32_t bh = (uint32_t)row / (uint32_t)p.Sq, b = bh / (uint32_t)p.H;
        at = b * p.os[0] + (bh - b * p.H) * p.os[1] + ((uint32_t)row - bh * p.Sq) * p.os[2];
    } else {
        at = row / p.Sq / p.H * p.os[0] + row / p.Sq % p.H * p.os[1] + row % p.Sq * p.os[2];
    }
    at += dim * p.os[3];
#pragma unroll
    for (int e = 0; e < 4; e++) A[e] /= L;  // no visible key: 0/0 = NaN
    if (out_vec && sizeof(T) == 2 && !p.out_f32) {
        T four[4] = {from_float<T>(A[0]), from_float<T>(A[1]), from_float<T>(A[2]), from_float<T>(A[3])};
        uint2_t w;
        __builtin_memcpy(&w, four, 8);
        *(uint2_t *)((T *)p.out + at) = w;
    } else if (out_vec) {
        *(float4_t *)((float *)p.out + at) = A;
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) store_out<T>(p, at + e * p.os[3], A[e]);
    }
}

// ---- head_dim 129 .. 256 (Gemma-3's key length is 256) -------------------------------------------------------
// A wavefront cannot hold 256 dims of Q and O for 32 rows, so two wavefronts share the 32 rows: wavefront
// `hf` of the pair owns dims [128 hf, 128 hf + 128) of Q, K, V and O.  Per key tile each computes its half of
// the contraction S^T = K Q^T, the halves are exchanged through LDS (in the K tile's space, which is free by
// then) and added, both run the same softmax on the same sums, and each accumulates its half of O^T.
// Workgroup = 2 pairs = 64 query rows; K, V tiles of 32 keys x 256 dims (zero-padded above head_dim).
constexpr int PFW_DP = 256, PFW_DH = 128;

template <typename T>
__global__ __launch_bounds__(64 * PF32_WAVES, 2) void prefill_f32_wide_kernel(AttnParams p, int nqb) {
    request_arguments<AttnParams, int>();
    constexpr int BM = 64;
    constexpr int KP = PFW_DP * 4 + 16;
    constexpr int K_BYTES = PF32_BN * KP;
    constexpr int CPR = PFW_DP / 4;
    constexpr int NCH = PF32_BN * CPR / (64 * PF32_WAVES);
    static_assert(PF32_WAVES * 16 * 256 <= K_BYTES, "the score exchange must fit the K tile's space");
    __shared__ __attribute__((aligned(16))) char smem[2 * K_BYTES];
    auto lds_base = (__attribute__((address_space(3))) char *)smem;

    if (p.iv_bad && *p.iv_bad == p.bad_tag) return;  // the mask is not made of intervals: the general kernel takes the call
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int ln = lane & 31;
    const int h2 = lane >> 5;
    const int pr = wave >> 1;  // which 32 rows
    const int hf = wave & 1;   // which half of the dims
    const int d0 = PFW_DH * hf;

    // Packed form (at most 32 query rows, an even GQA group): the two pairs hold rows 0..31 of two query heads that share
    // a KV head, so both work on every tile the workgroup moves (with one head per workgroup the second pair has no
    // rows) and a few new rows on a long cache need half the workgroups.
    const int pack = p.pf_pack;
    const int heads = pack ? p.H / 2 : p.H;  // head units per batch entry
    const int bh_count = p.B * heads;
    const int nks = max(p.pf_nsplit, 1);
    const int ksplit = blockIdx.x % nks;  // which share of the keys (0 when the keys are not split over workgroups)
    const int id = blockIdx.x / nks;
    const int qb = nqb - 1 - id / bh_count;
    int rem = id % bh_count;
    const int b = rem / heads;
    int h = rem % heads;
    if (pack) h = 2 * h + pr;
    else if ((p.H & 7) == 0) h = (h & 7) * (p.H >> 3) + (h >> 3);
    const int g = h / p.G;
    // Rows of a tile beyond the sequence's own keys (kv_lens below the view's length: a ragged batch in one cache
    // allocation) are never fetched: what such rows hold, NaN included, must not reach the result as 0 x NaN in P . V.
    // (likewise the rows behind the last query's own position when the call says where its rows stand inside a longer
    // cache view: a causal descriptor with q_pos_offset + Sq below the view's length)
    int key_end = p.kv_lens ? min(p.Skv, max(p.kv_lens[b], 1)) : p.Skv;
    if (p.analytic && p.causal) key_end = (int)min((int64_t)key_end, max(p.q_pos_offset + p.Sq, (int64_t)1));

    const int q0 = pack ? 0 : qb * BM;
    const int qw0 = pack ? 0 : q0 + 32 * pr;
    const int query = qw0 + ln;
    RowBounds rb = row_bounds(p, b, q0, pack ? 32 : BM, qw0, lane);
    if (nks > 1) {  // this workgroup's share of the keys
        const int c_lo = ksplit * p.pf_chunk, c_hi = c_lo + p.pf_chunk;
        rb.lo_wg = max(rb.lo_wg, c_lo), rb.hi_wg = min(rb.hi_wg, c_hi);
        rb.lo_w = max(rb.lo_w, c_lo), rb.hi_w = min(rb.hi_w, c_hi);
        rb.full_lo_w = max(rb.full_lo_w, c_lo), rb.full_hi_w = min(rb.full_hi_w, c_hi);
        rb.klo = max(rb.klo, c_lo), rb.khi = min(rb.khi, c_hi);
    }
    const int lo_wg = rb.lo_wg, hi_wg = rb.hi_wg, lo_w = rb.lo_w, hi_w = rb.hi_w;
    const bool wave_has_rows = qw0 < p.Sq;

    float4_t qreg[PFW_DH / 8];
    {
        const int qrow = min(query, p.Sq - 1);
        const T *qp = (const T *)p.q + b * p.qs[0] + h * p.qs[1] + (int64_t)qrow * p.qs[2];
#pragma unroll
        for (int kc = 0; kc < PFW_DH / 8; kc++) {
            const int dim = d0 + 8 * kc + 4 * h2;
            qreg[kc] = dim < p.D ? load4(qp + dim) : float4_t{0.f, 0.f, 0.f, 0.f};
        }
    }
    const T *kg = (const T *)p.k + b * p.ks[0] + g * p.ks[1];
    const T *vg = (const T *)p.v + b * p.vs[0] + g * p.vs[1];

    float16_t o[PFW_DH / 32];
#pragma unroll
    for (int db = 0; db < PFW_DH / 32; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[db][r] = 0.0f;
    float m = -INFINITY, l = 0.0f;
    const float scale2 = p.scale * PF32_LOG2E;

    // K and V take turns in one set of staging registers: V(j) is in flight while K(j) is multiplied, K(j+1)
    // while V(j) is
    float4_t st[NCH];
    auto load_rows = [&](const T *base, const int64_t row_stride, int j0) {
#pragma unroll
        for (int i = 0; i < NCH; i++) {
            const int cid = tid + 64 * PF32_WAVES * i;
            const int row = cid / CPR, col = cid % CPR;
            const int key = min(j0 + row, key_end - 1);
            st[i] = col * 4 < p.D ? load4(base + (int64_t)key * row_stride + col * 4) : float4_t{0.f, 0.f, 0.f, 0.f};
        }
    };
    auto store_rows = [&](int lds_off) {
#pragma unroll
        for (int i = 0; i < NCH; i++) {
            const int cid = tid + 64 * PF32_WAVES * i;
            const int row = cid / CPR, col = cid % CPR;
            *LDS32_PTR(float4_t, lds_off + row * KP + col * 16) = st[i];
        }
    };

    const int j_begin = (lo_wg / PF32_BN) * PF32_BN;
    if (j_begin < hi_wg) load_rows(kg, p.ks[2], j_begin);

    // every wavefront passes the same four barriers per tile, whether or not its rows see the tile
    for (int j0 = j_begin; j0 < hi_wg; j0 += PF32_BN) {
        store_rows(0);                    // K(j); its space is free since the last barrier of the previous tile
        load_rows(vg, p.vs[2], j0);       // V(j), needed after the softmax
        lds_barrier();
        const bool tile_visible = wave_has_rows && j0 < hi_w && j0 + PF32_BN > lo_w;  // the same for both halves

        // this half of S^T: contraction step (kc, i) uses dim d0 + 8 kc + 4 h2 + i on both operands
        float16_t s;
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = 0.0f;
        if (tile_visible) {
#pragma unroll
            for (int kc = 0; kc < PFW_DH / 8; kc++) {
                const float4_t a = *LDS32_PTR(float4_t, ln * KP + (d0 + 8 * kc + 4 * h2) * 4);
#pragma unroll
                for (int i = 0; i < 4; i++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], qreg[kc][i], s, 0, 0, 0);
            }
        }
        lds_barrier();  // the K tile has been read: its space takes the exchange
        if (tile_visible) {
#pragma unroll
            for (int r = 0; r < 16; r++) *LDS32_PTR(float, wave * 4096 + r * 256 + lane * 4) = s[r];
        }
        lds_barrier();
        if (tile_visible) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float other = *LDS32_PTR(float, (wave ^ 1) * 4096 + r * 256 + lane * 4);
                s[r] = hf == 0 ? s[r] + other : other + s[r];  // low + high half on both wavefronts: identical sums
            }
        }
        store_rows(K_BYTES);              // V(j); every wavefront is past P.V of the previous tile
        if (j0 + PF32_BN < hi_wg) load_rows(kg, p.ks[2], j0 + PF32_BN);  // K(j+1)
        lds_barrier();                    // V(j) visible, the exchange has been read
        if (!tile_visible) continue;

        // element r is key j0 + 8 (r / 4) + 4 h2 + r % 4 for query `query`
        if (!(j0 >= rb.full_lo_w && j0 + PF32_BN <= rb.full_hi_w)) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int key = j0 + 8 * (r >> 2) + 4 * h2 + (r & 3);
                s[r] = (key >= rb.klo && key < rb.khi) ? s[r] : -INFINITY;
            }
        }

        float mx = s[0];
#pragma unroll
        for (int r = 1; r < 16; r++) mx = fmaxf(mx, s[r]);
        mx = half_swap_max32(mx);
        const float m_new = fmaxf(m, mx * scale2);
        const float m_safe = (m_new == -INFINITY) ? 0.0f : m_new;
        const float corr = __builtin_amdgcn_exp2f(m - m_safe);
        m = m_new;
        float psum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], scale2, -m_safe));
            psum += s[r];
        }
        l = l * corr + psum;
#pragma unroll
        for (int db = 0; db < PFW_DH / 32; db++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[db][r] *= corr;

        // this half of O^T += V^T . P^T
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int krow = 8 * (r >> 2) + 4 * h2 + (r & 3);
#pragma unroll
            for (int db = 0; db < PFW_DH / 32; db++) {
                const float a = *LDS32_PTR(float, K_BYTES + krow * KP + (d0 + 32 * db + ln) * 4);
                o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, s[r], o[db], 0, 0, 0);
            }
        }
    }

    const float l_tot = half_swap_sum32(l);
    if (nks > 1) {
        // park this share's state (each wavefront of the pair its half of the dims); the merge kernel normalises
        if (query < p.Sq) {
            float *ws = p.partials + ((((int64_t)b * p.H + h) * p.Sq + query) * nks + ksplit) * p.pf_pitch;
#pragma unroll
            for (int db = 0; db < PFW_DH / 32; db++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int dim = d0 + 32 * db + 8 * (r >> 2) + 4 * h2 + (r & 3);
                    if (dim < p.D) ws[dim] = o[db][r];
                }
            if (hf == 0 && h2 == 0) {
                ws[p.D] = m;
                ws[p.D + 1] = l_tot;
            }
        }
        return;
    }
    if (query < p.Sq) {
        const int64_t ob = b * p.os[0] + h * p.os[1] + (int64_t)query * p.os[2];
#pragma unroll
        for (int db = 0; db < PFW_DH / 32; db++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int dim = d0 + 32 * db + 8 * (r >> 2) + 4 * h2 + (r & 3);
                if (dim < p.D) store_out<T>(p, ob + dim * p.os[3], o[db][r] / l_tot);  // no visible key: 0/0 = NaN like the reference
            }
    }
}

template <typename T>
static int launch_merge_t(const AttnParams &p, hipStream_t stream);

// query heads that share one workgroup of the wide-head kernel (0: one head, up to 64 rows)
static int prefill_f32_wide_pack(int G, int Sq, int D) { return (D > 128 && Sq <= 32 && G >= 2 && G % 2 == 0) ? 2 : 0; }

static int no_wide_bias() {
    set_error("prefill f32: a mask tensor without its interval form is not supported above head_dim 128");
    return FHIP_ERR_UNSUPPORTED;
}

template <typename T>
static int launch_wide(const AttnParams &p_in, hipStream_t stream) {
    if (p_in.mask && !p_in.iv) return no_wide_bias();
    AttnParams p = p_in;
    p.pf_pack = prefill_f32_wide_pack(p.G, p.Sq, p.D);
    const int nqb = p.pf_pack ? 1 : (p.Sq + 63) / 64;
    const long blocks = (long)nqb * p.B * (p.pf_pack ? p.H / 2 : p.H) * (p.pf_nsplit > 1 ? p.pf_nsplit : 1);
    if (blocks > 0x7fffffffL) {
        set_error("prefill f32: too many workgroups (%ld)", blocks);
        return FHIP_ERR_UNSUPPORTED;
    }
    FHIP_LAUNCH_MAIN(prefill_f32_wide_kernel<T>, dim3((unsigned)blocks), dim3(64 * PF32_WAVES), stream, p, p, nqb);
    FHIP_HIP_CHECK(hipGetLastError());
    if (p.pf_nsplit > 1) return launch_merge_t<T>(p, stream);
    return FHIP_OK;
}

template <typename T>
static int launch_merge_t(const AttnParams &p, hipStream_t stream) {
    const int64_t rows = (int64_t)p.B * p.H * p.Sq;
    const int lpr = p.D <= 64 ? 16 : p.D <= 128 ? 32 : 64, per = 256 / lpr;
    // rows of the result written in pieces of four elements
    const int oeb = sizeof(T) == 4 || p.out_f32 ? 4 : 2;
    int out_vec = p.os[3] == 1 && (uintptr_t)p.out % (4 * oeb) == 0;
    for (int i = 0; i < 3; i++)
        if (p.os[i] % 4 != 0) out_vec = 0;
    const dim3 grid((unsigned)((rows + per - 1) / per));
    if (lpr == 16) hipLaunchKernelGGL((prefill_f32_merge_kernel<T, 16>), grid, dim3(256), 0, stream, p, out_vec);
    else if (lpr == 32) hipLaunchKernelGGL((prefill_f32_merge_kernel<T, 32>), grid, dim3(256), 0, stream, p, out_vec);
    else hipLaunchKernelGGL((prefill_f32_merge_kernel<T, 64>), grid, dim3(256), 0, stream, p, out_vec);
    FHIP_HIP_CHECK(hipGetLastError());
    return FHIP_OK;
}

int launch_prefill_merge(const AttnParams &p, fhip_dtype dtype, hipStream_t stream) {
    if (dtype == FHIP_F16) return launch_merge_t<half_t>(p, stream);
    if (dtype == FHIP_BF16) return launch_merge_t<bf16_t>(p, stream);
    return launch_merge_t<float>(p, stream);
}

template <typename T, int MODE>
static int launch_rows(const AttnParams &p, hipStream_t stream) {
    constexpr int BM = 32 * PF32_WAVES;
    const int nqb = (p.Sq + BM - 1) / BM;
    const long blocks = (long)nqb * p.B * p.H * (p.pf_nsplit > 1 ? p.pf_nsplit : 1);
    if (blocks > 0x7fffffffL) {
        set_error("prefill f32: too many workgroups (%ld)", blocks);
        return FHIP_ERR_UNSUPPORTED;
    }
    dim3 grid((unsigned)blocks), block(64 * PF32_WAVES);
    switch ((p.D + 31) / 32 * 32) {  // the kernel's D is head_dim rounded up to a multiple of 32
        case 32: FHIP_LAUNCH_MAIN((prefill_f32_kernel<T, 32, MODE>), grid, block, stream, p, p, nqb); break;
        case 64: FHIP_LAUNCH_MAIN((prefill_f32_kernel<T, 64, MODE>), grid, block, stream, p, p, nqb); break;
        case 96:
            if constexpr (MODE != PF32_EITHER) FHIP_LAUNCH_MAIN((prefill_f32_kernel<T, 96, MODE>), grid, block, stream, p, p, nqb);
            break;
        case 128:
            if constexpr (MODE != PF32_EITHER) FHIP_LAUNCH_MAIN((prefill_f32_kernel<T, 128, MODE>), grid, block, stream, p, p, nqb);
            break;
        default: set_error("prefill f32 kernel: head_dim %d is not a multiple of 4 up to 128", p.D); return FHIP_ERR_UNSUPPORTED;
    }
    FHIP_HIP_CHECK(hipGetLastError());
    return FHIP_OK;
}

// Shares of the keys: the fewest within 2 % of the least time, where that is less than `gain` of the time of `ordinary` ones.  The times
// are those of a number's quickest form, although f32 tensors keep the form of the workgroups' numbers unless it is 10 % better
// (prefill_f32_terms_form): in the form that runs the model takes fewer or more shares for a few per cent that it is off itself (60 calls whose shares
// differ: 0.92 to 1.20 of the time, 1.03 in the mean; 8/4 heads at 64, 162 rows on 390 keys 12.8 -> 14.6 us).  Only causal chunks of more than a
// round, which lose by half a round too many, go by the form that runs (prefill_f32_unsplit_time).  16-bit tensors have one form.
static long shares_of_least_time(const TermsCall &c, long ordinary, double gain) {
    constexpr int SHARES[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 28, 32, 40, 48};
    const long units = (long)c.G * ((c.Sq + 31) / 32);
    double times[sizeof(SHARES) / sizeof(SHARES[0])], least = 0.0;
    int tried = 0;
    const TermsForm whole = prefill_f32_terms_form(c, 1);
    const bool by_form = prefill_f32_unsplit_time(c, whole) < prefill_f32_terms_time(c, whole, 1);
    auto time_in = [&](TermsForm form, int n) { return n > 1 ? prefill_f32_terms_time(c, form, n) : prefill_f32_unsplit_time(c, form); };
    for (const int n : SHARES) {
        // (shares that make three rounds of the smallest workgroups gain nothing more)
        if (n > 1 && (c.Skv / n < 64 || prefill_f32_workspace_bytes(c.B, c.Hkv * c.G, c.Sq, c.D, n) > ((size_t)64 << 20) ||
                      (n - 1) * (long)c.B * c.Hkv * units > 6L * c.cus))
            break;
        // (what parking and merging alone takes grows with n)
        if (n > 1 && prefill_f32_merge_time(c, n) > 1.02 * least) break;
        times[tried] = time_in(by_form ? prefill_f32_terms_form(c, n) : prefill_f32_terms_quickest(c, n), n);
        if (tried == 0 || times[tried] < least) least = times[tried];
        tried++;
    }
    for (int i = 0; i < tried; i++) {
        if (times[i] > 1.02 * least) continue;
        return times[i] < gain * time_in(prefill_f32_terms_form(c, (int)ordinary), (int)ordinary) ? SHARES[i] : ordinary;
    }
    return ordinary;
}

// Time in us of an unsplit call of more than 64 rows above head_dim 128 on the f32 matrix instruction (launch_wide): 64-row workgroups that
// walk their rows' keys, two on a CU beyond one each.  Its tiles take longer than the terms kernel's, but its workgroups start sooner
// and see fewer keys beside a window's: short prompts and narrow windows (us there and in terms, head_dim 256: 95 rows of 12/12 heads
// 22.6 and 27.1, three sequences of 77 of 10/2 22.6 and 27.8, 832 of 12/12 under a window of 134 49 and 62; over 50 random such calls
// 0.94 of the time in terms).  9 % off in the mean square over 206 calls of up to 13 tiles.
static double wide_f32_time(const TermsCall &c) {
    const int keys = c.window > 0 && c.window < c.Skv - 64 ? (int)c.window + 64 : c.Skv;
    const double tile = c.D <= 192 ? 5.4 : c.uneven ? 5.75 : 6.2;
    const long wgs = (long)c.B * c.Hkv * c.G * ((c.Sq + 63) / 64);
    return (c.D <= 192 ? 8.5 : 6.0) + tile * ((keys + 31) / 32) * std::max(1.0, (double)wgs / c.cus);
}

// Few query rows on a long cache (a new chat turn, a prompt fed in pieces): the grid of query blocks alone leaves
// most CUs idle, so the keys are split over workgroups as well.
void prefill_f32_plan(int B, int H, int G, int Sq, int Skv, int D, bool f32, bool causal, bool causal_square, bool uneven, int64_t window,
                      bool unknown_lengths, int compute_units, int *nsplit, int *chunk) {
    *nsplit = 1;
    *chunk = Skv;
    if (D <= 128) {
        // attn_prefill_f32_terms.hip, whose forms with key groups give a CU eight wavefronts in one workgroup: one workgroup
        // per CU, shares of at least 256 keys, or 128 while 256-key shares of all units are fewer than the CUs.  (The same
        // for a causal descriptor and for a mask tensor: a square prompt keeps its plan, and with it its bits.)
        const bool few_rows = 2L * Sq <= Skv;
        const long units = (long)G * ((Sq + 31) / 32), kv_heads = (long)B * (H / G);
        long most = Skv / 256;
        if (few_rows && most * kv_heads * units < compute_units) most = Skv / 128;
        auto shares = [&](int U) {
            const long wgs = kv_heads * ((units + U - 1) / U);
            if (wgs == 0 || 2 * wgs > compute_units) return 1L;
            const long want = compute_units / wgs;
            return want < most ? want : most;
        };
        // Workgroups of two units, or above head_dim 64 of four, whose shares are twice as many: for few rows, and from 768 keys
        // on (causal, D = 128: 832 rows of 16/4 heads 50 us in two shares, 55 unsplit; 704 rows 45 and 48; 768 rows of 8/2 heads 33
        // in three, 38 in two shares for two units each).  Shorter prompts if they come to three shares of 160 keys, or of 128
        // where there is room for four: 640 rows of 16/4 heads 44.7 -> 39.1, 512 rows 33.7 -> 32.3, 384 rows of 8/2 heads 29.1 ->
        // 22.0; but two batches of 12 heads at D = 96 take 27.8 in three shares of 128 keys against 25.0 unsplit (384 rows), and
        // 41 in two shares against 37 (640 rows).
        long ns = shares(D > 64 && (few_rows || Skv >= 768) ? 4 : 2);
        if (D > 64 && !few_rows && Skv < 768) {
            const long most_before = most, wgs = kv_heads * ((units + 3) / 4);
            most = Skv / (4 * wgs <= compute_units ? 128 : 160);
            const long of_four = shares(4);
            if (of_four >= 3) ns = of_four;
            most = most_before;
        }
        // By this rule a call asks for at most 16 MiB of partials.  Only full grids of four-unit workgroups (256 x 128 rows) are beyond that:
        // 32, 64, 128, 256 or 512 rows of 32/8 heads at D = 128, and up to seven rows fewer.  They take half the shares on workgroups
        // of half the units, the workspace that such calls have always had, and more time for it: on 8192 keys 32 rows 49 us (40 in
        // twice the shares), 64 rows 79 (56), 128 rows 128 (96), 256 rows 244 (172), 512 rows 463 (327).
        constexpr size_t MOST_PARTIALS = (size_t)16 << 20;
        if (few_rows && D > 64 && prefill_f32_workspace_bytes(B, H, Sq, D, (int)ns) > MOST_PARTIALS) ns = shares(2);
        // More than 128 rows that see about the same keys (chunks, images): the shares of least time, where that is 5 % less than the
        // rule's (shares_gain); at most 64 MiB of partials (us a call: two sequences of 275 rows of 32/8
        // heads at 64 on 2911 keys 116 -> 92; 16 heads without a mask, 1156 rows at 128 148 -> 80, 2506 366 -> 285, 1147 at 80 109 -> 59; over 90
        // random calls the time is 0.91, the worst 1.03 of the rule's).  Square prompts to 768 keys keep the rule, masked or not.
        if (!uneven && Sq > 128 && (few_rows || Skv > 768)) ns = shares_of_least_time({B, H / G, G, Sq, Skv, D, compute_units, false, window, f32, causal}, ns < 2 ? 1 : ns, shares_gain(unknown_lengths));
        if (ns < 2) return;
        const long c = ((Skv + ns - 1) / ns + 31) / 32 * 32;
        *chunk = (int)c;
        *nsplit = (int)((Skv + c - 1) / c);
        return;
    }
    if (f32 && Sq > 64) {
        // Head dims above 128 in the terms kernel: the shares of least time (us, 16/4 heads at 256 causal, in one share and in
        // the shares taken: 148 rows on 3510 keys 584 -> 80, 300 on 700 128 -> 49, 1000 on 1000 182 -> 93, 2000 on 2000 347 -> 235; 2048 on 2048 stays at 355, its two shares
        // would be more than 64 MiB of partials).
        const TermsCall call = {B, H / G, G, Sq, Skv, D, compute_units, uneven, window, true, causal};
        const long ns = shares_of_least_time(call, 1, shares_gain(false));
        if (ns < 2 || wide_f32_time(call) < prefill_f32_terms_time(call, {4, 1}, (int)ns)) return;
        const long c = ((Skv + ns - 1) / ns + 31) / 32 * 32;
        *chunk = (int)c;
        *nsplit = (int)((Skv + c - 1) / c);
        return;
    }
    // Up to 64 rows, and 16-bit rows that only the kernel of this file takes (head dims not a multiple of 8): down to 512 keys per share, until there are about two workgroups per CU.  Square causal calls are
    // left alone (their shares would be uneven, and they fill the chip from 1024 rows on).
    if (causal_square) return;
    const int pack = prefill_f32_wide_pack(G, Sq, D);
    const long wgs = pack ? (long)B * (H / 2) : (long)B * H * ((Sq + 63) / 64);
    if (wgs > compute_units) return;  // the query blocks alone keep at least half the chip busy (two workgroups per CU)
    const long want = (2L * compute_units + wgs - 1) / wgs;
    // Shares of at least 512 keys (256 in the packed form, which has half the workgroups); while that leaves CUs without
    // a workgroup, down to 256 and then 128 keys: a workgroup alone on its CU spends most of a tile waiting for the
    // tile's rows (~7 us per 32-key tile), so more, shorter workgroups win until the chip is full (f32, B1: head_dim 256,
    // 2048 keys, 9 rows 55 -> 36 us).  Shorter shares than needed merge too often (head_dim 256, B1 x 8192 keys, 32 rows: 84 us with
    // 256 shares of 8 tiles, 101 us with 512 of 4).
    long most = Skv / (pack ? 256 : 512);
    // (only for calls that are clearly a few rows on a longer cache: a square prompt masked by a tensor keeps the plan
    // of its analytic twin, and with it the same bits)
    const bool few_rows = 2L * Sq <= Skv;
    if (few_rows && (want < most ? want : most) * wgs < compute_units) most = Skv / 256;
    if (few_rows && (want < most ? want : most) * wgs < compute_units) most = Skv / 128;
    long ns = want < most ? want : most;
    if (ns < 2) return;
    long c = (Skv + ns - 1) / ns;
    c = (c + 31) / 32 * 32;
    *chunk = (int)c;
    *nsplit = (int)((Skv + c - 1) / c);
}

size_t prefill_f32_workspace_bytes(int B, int H, int Sq, int D, int nsplit) {
    if (nsplit <= 1) return 0;
    return (size_t)B * H * Sq * nsplit * (size_t)(D + 2) * sizeof(float);
}

// Head dims above 128 in f32: the terms kernel, but for
//  - up to 64 rows whose shares leave CUs without a workgroup of launch_wide's, on up to 2048 keys, or above 192 dims half of the CUs: a
//    workgroup alone on its CU takes longer to split its first tile and Q into terms than the f32 instruction takes for both
//    (us, head_dim 256, here and in terms: 9 rows of 16/4 heads on 2048 keys 34.7 and 37.3, 33 rows on 1000 39.6 and 43.0, 16 of 4/1 on 3299
//    39.1 and 41.2; 64 rows of 4 heads on 4096 50.2 and 41.1, 17 rows of 32/8 heads on 8192 108 and 70);
//  - up to 64 rows whose heads leave half of the terms kernel's units empty, so that it has as many workgroups as launch_wide (40 to 50 rows of
//    16/16 heads on 1829 keys 73.7 and 78.8, of 32/32 on 3286 283 and 306);
//  - more rows that see few keys, unsplit (wide_f32_time).
static bool wide_in_terms(const AttnParams &p) {
    const int cus = p.cus > 0 ? p.cus : 256;
    const long ns = p.pf_nsplit > 1 ? p.pf_nsplit : 1;
    if (p.Sq > 64) {
        const TermsCall c = prefill_f32_terms_call(p);
        return ns > 1 || prefill_f32_terms_time(c, {4, 1}, 1) <= wide_f32_time(c);
    }
    const long wgs = (long)p.B * (prefill_f32_wide_pack(p.G, p.Sq, p.D) ? p.H / 2 : p.H);
    const long of_units = (long)p.B * p.Hkv * ((p.G * ((p.Sq + 31) / 32) + 3) / 4);
    return of_units < wgs && (wgs * ns >= cus || (p.Skv > 2048 && (p.D <= 192 || 2 * wgs * ns >= cus)));
}

template <typename T>
static int launch_prefill_f32_t(const AttnParams &p, hipStream_t stream) {
    if (p.D > 128 && !(sizeof(T) == 4 && wide_in_terms(p) && prefill_f32_terms_takes(p))) return launch_wide<T>(p, stream);
    if (p.D > 128 && p.mask && !p.iv) return no_wide_bias();
    const int mode = !p.mask ? PF32_INTERVALS : !p.iv && !p.iv_either ? PF32_BIAS : p.iv_either ? PF32_EITHER : PF32_INTERVALS;
    if (mode == PF32_EITHER && p.D > 64) {
        set_error("internal: the two-form f32 kernel takes head_dim <= 64");
        return FHIP_ERR_UNSUPPORTED;
    }
    int rc;
    if (prefill_f32_terms_takes(p)) {
        // 6 / 16 of this file's matrix time for the same precision (4096 x 4096 causal, D = 128: 1150 -> 700 us)
        rc = launch_prefill_f32_terms(p, sizeof(T) == 4 ? FHIP_F32 : std::is_same<T, half_t>::value ? FHIP_F16 : FHIP_BF16, mode, stream);
    } else {
        rc = mode == PF32_EITHER ? launch_rows<T, PF32_EITHER>(p, stream)
             : mode == PF32_BIAS ? launch_rows<T, PF32_BIAS>(p, stream)
                                 : launch_rows<T, PF32_INTERVALS>(p, stream);
    }
    if (rc || p.pf_nsplit <= 1) return rc;
    return launch_merge_t<T>(p, stream);
}

int launch_prefill_f32(const AttnParams &p, fhip_dtype dtype, hipStream_t stream) {
    if (dtype == FHIP_F16) return launch_prefill_f32_t<half_t>(p, stream);
    if (dtype == FHIP_BF16) return launch_prefill_f32_t<bf16_t>(p, stream);
    return launch_prefill_f32_t<float>(p, stream);
}

}  // namespace fhip
